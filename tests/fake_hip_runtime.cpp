// fake_hip_runtime.cpp - the HIP calls and kernel launches of csrc/ntc_hip_api.cpp on host memory, for tests of its host
// code without a GPU: any call can be made to fail, and a launch stays outstanding until its stream is waited for.
// Linked with that file's object in the place of libamdhip64 and of the kernels; tests/test_host_failures.py drives it.
#include <hip/hip_runtime.h>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include "../rtxntc-library_amd/csrc/ntc_decode_kernel.h"

using namespace ntc_hip_dev;

namespace {
struct Stream { int outstanding = 0; };
struct Event { Stream* stream = nullptr; };
Stream g_null;
std::set<void*> g_memory;
std::map<std::string, int> g_failIn;       // calls until the one that fails
hipError_t g_last = hipSuccess;
std::string g_launches;                    // names of the launches and of the stream waits, a line each
int g_dropRows = 0, g_dirtyCounters = 0, g_nullStreamUses = 0;

Stream* of(hipStream_t s)
{
    if (!s) ++g_nullStreamUses;
    return s ? reinterpret_cast<Stream*>(s) : &g_null;
}
hipError_t outcome(char const* name, hipError_t error = hipErrorOutOfMemory)
{
    auto const at = g_failIn.find(name);
    if (at == g_failIn.end() || --at->second > 0) return hipSuccess;
    g_failIn.erase(at);
    return g_last = error;
}
hipError_t launched(char const* name, hipStream_t stream)
{
    if (hipError_t const e = outcome(name, hipErrorLaunchFailure)) return e;
    ++of(stream)->outstanding;
    g_launches += std::string(name) + '\n';
    return hipSuccess;
}
hipError_t allocate(char const* name, void** p, size_t bytes)
{
    if (hipError_t const e = outcome(name)) return e;
    *p = std::malloc(bytes ? bytes : 1);
    std::memset(*p, 0xA5, bytes);          // what memory holds is nobody's promise
    g_memory.insert(*p);
    return hipSuccess;
}
hipError_t release(void* p)
{
    if (!g_memory.erase(p)) return g_last = hipErrorInvalidValue;
    std::free(p);
    return hipSuccess;
}
} // namespace

extern "C" {

// ---- the test's side
void fake_reset() { g_failIn.clear(); g_last = hipSuccess; g_dropRows = g_dirtyCounters = 0; }
void fake_fail(char const* name, int call) { g_failIn[name] = call; }
void fake_drop_rows(int count) { g_dropRows = count; }             // so many of the next loss launches store nothing
int fake_dirty_counters() { return g_dirtyCounters; }              // loss launches that found a counter other than zero
int fake_null_stream_uses() { return g_nullStreamUses; }
char const* fake_launches() { return g_launches.c_str(); }        // since the library was loaded
int fake_allocations() { return int(g_memory.size()); }
hipStream_t fake_last_loss_stream = nullptr;
int fake_outstanding() { return reinterpret_cast<Stream*>(fake_last_loss_stream)->outstanding; }

// ---- the runtime
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int)          // (a macro of the present structure's name)
{
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
char const* hipGetErrorName(hipError_t e) { return e == hipSuccess ? "hipSuccess" : "hipErrorOfTheTest"; }
hipError_t hipGetLastError() { hipError_t const e = g_last; g_last = hipSuccess; return e; }
hipError_t hipMalloc(void** p, size_t bytes) { return allocate("hipMalloc", p, bytes); }
hipError_t hipFree(void* p) { return p ? release(p) : hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { return allocate("hipHostMalloc", p, bytes); }
hipError_t hipHostFree(void* p) { return release(p); }
hipError_t hipHostGetDevicePointer(void** dev, void* host, unsigned)
{
    if (hipError_t const e = outcome("hipHostGetDevicePointer")) return e;
    *dev = host;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, void const*) { static char table[1 << 16]; *p = table; return hipSuccess; }
hipError_t hipMemcpy(void* d, void const* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, void const* s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t* s) { *s = reinterpret_cast<hipStream_t>(new Stream); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    if (hipError_t const e = outcome("hipStreamCreateWithFlags")) return e;
    return hipStreamCreate(s);
}
hipError_t hipStreamDestroy(hipStream_t s) { delete reinterpret_cast<Stream*>(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s)
{
    of(s)->outstanding = 0;
    g_launches += "complete\n";
    return outcome("hipStreamSynchronize", hipErrorLaunchFailure);
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    if (hipError_t const r = outcome("hipEventCreate")) return r;
    *e = reinterpret_cast<hipEvent_t>(new Event);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<Event*>(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { *reinterpret_cast<Event*>(e) = Event{ of(s) }; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e)
{
    if (Stream* const s = reinterpret_cast<Event*>(e)->stream) s->outstanding = 0;
    return outcome("hipEventSynchronize", hipErrorLaunchFailure);
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.f; return hipSuccess; }
hipError_t hipLaunchKernel(void const*, dim3, dim3, void**, size_t, hipStream_t s) { return g_last = launched("hipLaunchKernel", s); }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
void** __hipRegisterFatBinary(void const*) { static void* handle; return &handle; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, void const*, char*, char const*, unsigned, uint3*, uint3*, dim3*, dim3*, int*) {}
void __hipRegisterVar(void**, void*, char*, char const*, int, size_t, int, int) {}

} // extern "C"

// ---- the launchers
namespace ntc_hip_dev {
int compute_units_of_current_device() { return 256; }
hipError_t launch_fill(uint8_t* dst, uint8_t value, uint64_t bytes, hipStream_t s)
{
    if (hipError_t const e = launched("launch_fill", s)) return e;
    std::memset(dst, value, bytes);
    return hipSuccess;
}
// Channel c's sum is (c + 1) * width * height, in one group's row each; zeros in the other rows.
hipError_t launch_image_loss(uint16_t*, uint16_t const*, int width, int height, int, uint32_t, int, int, LossWorkspace const& work, hipStream_t s, hipEvent_t done)
{
    if (hipError_t const e = launched("launch_image_loss", s)) return e;
    fake_last_loss_stream = s;
    *reinterpret_cast<Event*>(done) = Event{ of(s) };
    for (uint32_t i = 0; i < kLossRows; ++i)
        if (work.counters[i] != 0) { ++g_dirtyCounters; break; }
    if (g_dropRows > 0) { --g_dropRows; return hipSuccess; }
    LossGrid const grid = image_loss_grid(width, height, 256);
    uint32_t const rows = (grid.x * grid.y + grid.groupSize - 1) / grid.groupSize;
    for (uint32_t r = 0; r < rows; ++r)
        for (int c = 0; c < NTC_HIP_DEV_MAX_CHANNELS; ++c) {
            double const sum = uint32_t(c) % rows == r ? double(c + 1) * width * height : 0.0;
            uint64_t bits;
            std::memcpy(&bits, &sum, 8);
            work.rows[r].words[2 * c] = uint64_t(work.serial) << 32 | (bits & 0xffffffffu);
            work.rows[r].words[2 * c + 1] = uint64_t(work.serial) << 32 | bits >> 32;
        }
    return hipSuccess;
}
hipError_t launch_color_tables(hipStream_t s) { return launched("launch_color_tables", s); }
hipError_t launch_transfer_tables(hipStream_t s) { return launched("launch_transfer_tables", s); }
hipError_t launch_read_channels(ReadChannelsArgs const&, hipStream_t s) { return launched("launch_read_channels", s); }
hipError_t launch_write_channels(WriteChannelsArgs const&, hipStream_t s) { return launched("launch_write_channels", s); }
hipError_t launch_resize_planar(uint16_t const*, int, int, uint16_t*, int, int, int, uint8_t const*, hipStream_t s) { return launched("launch_resize_planar", s); }
hipError_t launch_image_difference(ImageDifferenceArgs const&, hipStream_t s) { return launched("launch_image_difference", s); }
hipError_t launch_block_compress(BlockCompressArgs const&, int, hipStream_t s) { return launched("launch_block_compress", s); }
hipError_t launch_decode(int, MipTable const&, int, int, int, hipStream_t s) { return launched("launch_decode", s); }
hipError_t launch_decode_fp8(int, MipTable const&, int, int, int, Fp8Handoff, hipStream_t s) { return launched("launch_decode_fp8", s); }
hipError_t launch_queries(int, MipTable const&, int, DevQuery const*, uint64_t, uint16_t*, int, hipStream_t s) { return launched("launch_queries", s); }
hipError_t launch_queries_fp8(int, MipTable const&, int, DevQuery const*, uint64_t, uint16_t*, int, Fp8Handoff, hipStream_t s) { return launched("launch_queries_fp8", s); }
hipError_t launch_build_bricks(uint16_t const*, uint8_t*, int, int, int, hipStream_t s) { return launched("launch_build_bricks", s); }
hipError_t launch_selftest_mfma(int8_t const*, int8_t const*, int32_t*, hipStream_t s) { return launched("launch_selftest_mfma", s); }
hipError_t launch_selftest_mfma_f16(uint16_t const*, uint16_t const*, float const*, float*, int, hipStream_t s) { return launched("launch_selftest_mfma_f16", s); }
hipError_t launch_selftest_fp8_activation(uint16_t const*, uint16_t*, int, hipStream_t s) { return launched("launch_selftest_fp8_activation", s); }
int resident_workgroups_per_cu(int) { return 4; }
int resident_fp8_workgroups_per_cu() { return 4; }
int tiles_per_round(int) { return 8; }
int fp8_tiles_per_round() { return 8; }
int threads_per_workgroup(int) { return 256; }
int fp8_threads_per_workgroup() { return 256; }
} // namespace ntc_hip_dev
