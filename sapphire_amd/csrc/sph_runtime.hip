// Device, memory, stream and event entry points of the C ABI.
//
// The reference keeps one cuBLAS handle per (device, thread) and relies on the
// per-thread default stream (Sources/Sapphire/compute/dense/cuda/Gemm.cu:24-30,
// CMake/CompileOptions.cmake:227).  Here the same slot holds a HIP stream:
// every thread gets its own non-blocking stream per device, created on first
// use at the default priority and free for another thread when the thread
// ends, so no stream is destroyed while the runtime may be shutting down.
#include "sph_internal.h"
#include "sph_spgemm_plan.h"

#include <atomic>
#include <cstring>
#include <mutex>
#include <new>

namespace
{
constexpr int kMaxDevices = 16;

thread_local std::string tlsLastError;

// A stream of the library's own, with the staging block that calls on it have left behind.  Made once
// and never destroyed; the thread that has the stream takes and gives back the block, any thread may
// hand an idle one back to its pool.
struct OwnStream
{
    hipStream_t stream = nullptr;
    // (the rest under the mutex below)
    OwnStream* next = nullptr;  // of the device
    bool used = true;           // a thread has it
    void* block = nullptr;
    size_t bytes = 0;
    bool taken = false;  // by the call that runs
};

std::mutex gPoolMutex;
OwnStream* gStreams[kMaxDevices] = {};
size_t gBlockBytes[kMaxDevices] = {};  // of their blocks
int gComputeUnits[kMaxDevices] = {};
bool gPoolRetains[kMaxDevices] = {};
// (same mutex) the devices' default pools, and the library's own pools for the scratch blocks of
// its calls, created on first use and kept until the process ends
hipMemPool_t gDefaultPools[kMaxDevices] = {};
hipMemPool_t gScratchPools[kMaxDevices] = {};

struct ThreadSlots
{
    int device = 0;
    OwnStream* own[kMaxDevices] = {};
    hipStream_t borrowed[kMaxDevices] = {};
    hipStream_t capturing = nullptr;  // stream under capture, if any

    ~ThreadSlots()
    {
        std::lock_guard<std::mutex> lock(gPoolMutex);
        for (int d = 0; d < kMaxDevices; ++d)
            if (own[d] != nullptr)
                own[d]->used = false;
    }
};

thread_local ThreadSlots tlsSlots;
}  // namespace

namespace
{
std::atomic<uint64_t> gAllocations{0};
}

namespace sph
{
void CountAllocation()
{
    gAllocations.fetch_add(1, std::memory_order_relaxed);
}

// With a release threshold of zero, the default of a device's pool, every synchronisation hands
// freed blocks back to the driver, and the next call maps its staging anew: a CSR x CSR product of
// 65536 rows (139 MB of staging) that is waited for took 384 us, 87 us of them on the GPU (now
// 96 us; dense to CSR, 8192 x 4096, 58 -> 38 us).  So the blocks come from a pool of the
// library's own that keeps a bounded amount: the device's default pool belongs to the program,
// whose threshold and whose other users are left alone.  Where the program has the default pool
// keep at least as much itself (sph_malloc_async does), that pool is used.
constexpr uint64_t kScratchKept = 512ull << 20;

namespace
{
int ScratchPool(hipMemPool_t* pool)
{
    const int d = tlsSlots.device;
    std::lock_guard<std::mutex> lock(gPoolMutex);
    if (gDefaultPools[d] == nullptr)
        SPH_HIP_TRY(hipDeviceGetDefaultMemPool(&gDefaultPools[d], d));
    *pool = gDefaultPools[d];
    uint64_t keep = 0;  // the program may change it at any time
    SPH_HIP_TRY(hipMemPoolGetAttribute(*pool, hipMemPoolAttrReleaseThreshold, &keep));
    if (keep >= kScratchKept)
        return SPH_OK;
    if (gScratchPools[d] == nullptr)
    {
        hipMemPoolProps props{};
        props.allocType = hipMemAllocationTypePinned;
        props.handleTypes = hipMemHandleTypeNone;
        props.location.type = hipMemLocationTypeDevice;
        props.location.id = d;
        hipMemPool_t own = nullptr;
        SPH_HIP_TRY(hipMemPoolCreate(&own, &props));
        keep = kScratchKept;
        const hipError_t set = hipMemPoolSetAttribute(own, hipMemPoolAttrReleaseThreshold, &keep);
        if (set != hipSuccess)
        {
            (void)hipMemPoolDestroy(own);
            SPH_HIP_TRY(set);
        }
        gScratchPools[d] = own;
    }
    *pool = gScratchPools[d];
    return SPH_OK;
}

// The mutex is held: the stream's block goes back to its pool, behind the work that has used it.
hipError_t DropBlock(OwnStream& own)
{
    const hipError_t err = hipFreeAsync(own.block, own.stream);
    gBlockBytes[tlsSlots.device] -= own.bytes;
    own.block = nullptr;
    own.bytes = 0;
    return err;
}

// The idle blocks of the device go back to their pools: the calling thread's own, and those of streams
// that have nothing to do, whether another thread has them or none.  (A stream under capture is
// left alone: what is asked of it would become a part of the graph.)  `wait`: for the work that has
// used the thread's own block.
hipError_t DropIdleBlocks(bool wait)
{
    std::lock_guard<std::mutex> lock(gPoolMutex);
    for (OwnStream* s = gStreams[tlsSlots.device]; s != nullptr; s = s->next)
    {
        if (s->block == nullptr || s->taken)
            continue;
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        hipError_t err = hipStreamIsCapturing(s->stream, &status);
        if (err != hipSuccess)
            return err;
        if (status != hipStreamCaptureStatusNone)
            continue;
        const bool mine = s == tlsSlots.own[tlsSlots.device];
        if (!mine)
        {
            err = hipStreamQuery(s->stream);
            if (err != hipSuccess)
            {
                (void)hipGetLastError();  // not the next launch's error
                if (err == hipErrorNotReady)
                    continue;
                return err;
            }
        }
        err = DropBlock(*s);
        if (err == hipSuccess && (wait || !mine))
            err = hipStreamSynchronize(s->stream);  // (the pool has it back when the stream has come to that)
        if (err != hipSuccess)
            return err;
    }
    return hipSuccess;
}

// Idle blocks go back to the pools, those of the library's own pool to the driver.
hipError_t TrimScratch(bool wait)
{
    const hipError_t dropped = DropIdleBlocks(wait);
    if (dropped != hipSuccess)
        return dropped;
    std::lock_guard<std::mutex> lock(gPoolMutex);
    hipMemPool_t own = gScratchPools[tlsSlots.device];
    return own != nullptr ? hipMemPoolTrimTo(own, 0) : hipSuccess;
}

// An allocation that finds the device full is tried once more without the idle scratch blocks.
template <typename Alloc>
hipError_t AllocWithTrim(Alloc&& alloc)
{
    hipError_t err = alloc();
    if (err != hipErrorOutOfMemory)
        return err;
    (void)hipGetLastError();  // not the next launch's error
    if (TrimScratch(true) == hipSuccess)
        err = alloc();
    if (err == hipErrorOutOfMemory)
        (void)hipGetLastError();
    return err;
}
}  // namespace

namespace
{
// SPH_OK and a null *ptr when the device is full
int BlockFromPool(void** ptr, size_t bytes, hipStream_t stream)
{
    *ptr = nullptr;
    hipMemPool_t pool = nullptr;
    const int found = ScratchPool(&pool);
    if (found != SPH_OK)
        return found;
    const hipError_t err =
        AllocWithTrim([&] { return hipMallocFromPoolAsync(ptr, bytes, pool, stream); });
    if (err == hipErrorOutOfMemory)
    {
        *ptr = nullptr;
        return SPH_OK;
    }
    SPH_HIP_TRY(err);
    CountAllocation();
    return SPH_OK;
}
}  // namespace

int AllocScratch(void** ptr, size_t bytes, hipStream_t stream)
{
    const int taken = BlockFromPool(ptr, bytes, stream);
    if (taken == SPH_OK && *ptr == nullptr)
        return Fail(SPH_ERR_DEVICE, std::string("no room for a scratch block of ") +
                                        std::to_string(bytes) + " bytes: " +
                                        hipGetErrorString(hipErrorOutOfMemory));
    return taken;
}

// Taking a block from a pool and giving it back costs the host 8 us, more than two launches, and a
// product of a few thousand rows is over before that.  Its staging, up to 32 MiB, therefore stays with
// the stream it was taken for, if that is one of the library's own: a later call on the stream runs behind
// the one before, so it may use the block at once.  Per thread and device that is one block, for all
// of them together as much as the pool keeps; a thread that ends leaves it, with the stream, to the
// next.  8192 rows of 64 products, calls one after the other 21.3 -> 18.1 us (host 21.3 -> 13.7).
constexpr size_t kKeptBlock = 32u << 20;

int TakeStaging(void** ptr, size_t bytes, hipStream_t stream)
{
    const int d = tlsSlots.device;
    OwnStream* own = tlsSlots.own[d];
    bool keep = own != nullptr && stream == own->stream && bytes <= kKeptBlock;
    if (keep)
    {
        std::lock_guard<std::mutex> lock(gPoolMutex);
        keep = !own->taken;
        if (keep && own->block != nullptr && own->bytes >= bytes)
        {
            own->taken = true;
            *ptr = own->block;
            return SPH_OK;
        }
        if (keep && own->block != nullptr)
            SPH_HIP_TRY(DropBlock(*own));
        keep = keep && gBlockBytes[d] + kKeptBlock <= kScratchKept;
        if (keep)
            gBlockBytes[d] += kKeptBlock;  // until it is known what the block is
    }
    if (!keep)
        return BlockFromPool(ptr, bytes, stream);
    int taken = SPH_OK;
    const size_t got = TakeWithRoom(bytes, kKeptBlock, [&](size_t size) {
        taken = BlockFromPool(ptr, size, stream);
        return taken != SPH_OK || *ptr != nullptr;
    });
    std::lock_guard<std::mutex> lock(gPoolMutex);
    gBlockBytes[d] -= kKeptBlock;
    if (taken == SPH_OK && *ptr != nullptr)
    {
        own->block = *ptr;
        own->bytes = got;
        own->taken = true;
        gBlockBytes[d] += got;
    }
    return taken;
}

int GiveStaging(void* ptr, hipStream_t stream)
{
    OwnStream* own = tlsSlots.own[tlsSlots.device];
    if (own != nullptr)
    {
        std::lock_guard<std::mutex> lock(gPoolMutex);
        if (own->taken && ptr == own->block)
        {
            own->taken = false;
            return SPH_OK;
        }
    }
    SPH_HIP_TRY(hipFreeAsync(ptr, stream));
    return SPH_OK;
}

int Fail(int status, const std::string& msg)
{
    tlsLastError = msg;
    return status;
}

int CurrentDevice()
{
    return tlsSlots.device;
}

hipStream_t CurrentStream()
{
    const int d = tlsSlots.device;
    if (tlsSlots.borrowed[d] != nullptr)
        return tlsSlots.borrowed[d];
    if (tlsSlots.own[d] == nullptr)
    {
        {
            std::lock_guard<std::mutex> lock(gPoolMutex);
            OwnStream* idle = gStreams[d];
            while (idle != nullptr && idle->used)
                idle = idle->next;
            if (idle != nullptr)
            {
                idle->used = true;
                tlsSlots.own[d] = idle;
                return idle->stream;
            }
        }
        OwnStream* own = new (std::nothrow) OwnStream;
        hipError_t err = own != nullptr ? hipSetDevice(d) : hipErrorOutOfMemory;
        if (err == hipSuccess)
            err = hipStreamCreateWithFlags(&own->stream, hipStreamNonBlocking);
        if (err != hipSuccess)
        {
            delete own;
            Fail(SPH_ERR_DEVICE,
                 std::string("stream creation failed with ") + hipGetErrorString(err));
            return nullptr;
        }
        std::lock_guard<std::mutex> lock(gPoolMutex);
        own->next = gStreams[d];
        gStreams[d] = own;
        tlsSlots.own[d] = own;
    }
    return tlsSlots.own[d]->stream;
}

bool Capturing()
{
    return tlsSlots.capturing != nullptr;
}

int ComputeUnits()
{
    const int d = tlsSlots.device;
    if (gComputeUnits[d] == 0)
    {
        int cu = 0;
        if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, d) !=
                hipSuccess ||
            cu <= 0)
            cu = 256;
        gComputeUnits[d] = cu;
    }
    return gComputeUnits[d];
}
}  // namespace sph

#define SPH_STREAM_OR_FAIL(var)                                                \
    hipStream_t var = ::sph::CurrentStream();                                  \
    if (var == nullptr)                                                        \
    return SPH_ERR_DEVICE

extern "C" {

const char* sph_last_error(void)
{
    return tlsLastError.c_str();
}

int sph_device_count(int* count)
{
    SPH_REQUIRE(count != nullptr, "count is null");
    int n = 0;
    const hipError_t err = hipGetDeviceCount(&n);
    if (err != hipSuccess)
    {
        *count = 0;
        return sph::Fail(SPH_ERR_DEVICE, std::string("hipGetDeviceCount failed with ") +
                                             hipGetErrorString(err));
    }
    *count = n;
    return SPH_OK;
}

int sph_set_device(int deviceId)
{
    SPH_REFUSE_WHILE_CAPTURING();
    int n = 0;
    const int rc = sph_device_count(&n);
    if (rc != SPH_OK)
        return rc;
    // Memory.cpp:14-28: an id at or beyond the device count is refused
    if (deviceId < 0 || deviceId >= n || deviceId >= kMaxDevices)
        return sph::Fail(SPH_ERR_INVALID,
                         "sph_set_device - deviceId exceeds number of available devices");
    SPH_HIP_TRY(hipSetDevice(deviceId));
    tlsSlots.device = deviceId;
    return SPH_OK;
}

int sph_get_device(int* deviceId)
{
    SPH_REQUIRE(deviceId != nullptr, "deviceId is null");
    *deviceId = tlsSlots.device;
    return SPH_OK;
}

int sph_device_info(int deviceId, SphDeviceInfo* info)
{
    SPH_REQUIRE(info != nullptr, "info is null");
    hipDeviceProp_t prop;
    SPH_HIP_TRY(hipGetDeviceProperties(&prop, deviceId));
    std::memset(info, 0, sizeof(*info));
    std::strncpy(info->name, prop.name, sizeof(info->name) - 1);
    std::strncpy(info->arch, prop.gcnArchName, sizeof(info->arch) - 1);
    info->computeUnits = prop.multiProcessorCount;
    info->clockMHz = prop.clockRate / 1000;
    info->memoryClockMHz = prop.memoryClockRate / 1000;
    info->memoryBusWidthBits = prop.memoryBusWidth;
    info->ldsBytesPerBlock = static_cast<int>(prop.sharedMemPerBlock);
    info->l2Bytes = prop.l2CacheSize;
    info->totalMemoryBytes = prop.totalGlobalMem;
    info->wavefrontSize = prop.warpSize;
    return SPH_OK;
}

int sph_malloc(void** ptr, size_t bytes)
{
    SPH_REFUSE_WHILE_CAPTURING();
    SPH_REQUIRE(ptr != nullptr, "ptr is null");
    SPH_HIP_TRY(hipSetDevice(tlsSlots.device));
    ::sph::CountAllocation();
    SPH_HIP_TRY(sph::AllocWithTrim([&] { return hipMalloc(ptr, bytes); }));
    return SPH_OK;
}

int sph_free(void* ptr)
{
    SPH_REFUSE_WHILE_CAPTURING();
    SPH_HIP_TRY(hipFree(ptr));
    return SPH_OK;
}

int sph_malloc_async(void** ptr, size_t bytes)
{
    SPH_REFUSE_WHILE_CAPTURING();
    SPH_REQUIRE(ptr != nullptr, "ptr is null");
    SPH_STREAM_OR_FAIL(stream);
    const int d = tlsSlots.device;
    {
        // freed blocks stay in the device's pool instead of going back to the driver
        std::lock_guard<std::mutex> lock(gPoolMutex);
        if (!gPoolRetains[d])
        {
            hipMemPool_t pool = nullptr;
            SPH_HIP_TRY(hipDeviceGetDefaultMemPool(&pool, d));
            uint64_t keep = ~0ull;
            SPH_HIP_TRY(hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep));
            gPoolRetains[d] = true;
        }
    }
    ::sph::CountAllocation();
    SPH_HIP_TRY(sph::AllocWithTrim(
        [&] { return hipMallocAsync(ptr, bytes != 0 ? bytes : 1, stream); }));
    return SPH_OK;
}

int sph_free_async(void* ptr)
{
    SPH_REFUSE_WHILE_CAPTURING();
    if (ptr == nullptr)
        return SPH_OK;
    SPH_STREAM_OR_FAIL(stream);
    SPH_HIP_TRY(hipFreeAsync(ptr, stream));
    return SPH_OK;
}

int sph_allocation_count(uint64_t* count)
{
    SPH_REQUIRE(count != nullptr, "count is null");
    *count = gAllocations.load(std::memory_order_relaxed);
    return SPH_OK;
}

int sph_mem_pool_trim(void)
{
    SPH_REFUSE_WHILE_CAPTURING();
    SPH_HIP_TRY(sph::TrimScratch(false));  // (first: an idle block may be of either pool)
    hipMemPool_t pool = nullptr;
    SPH_HIP_TRY(hipDeviceGetDefaultMemPool(&pool, tlsSlots.device));
    SPH_HIP_TRY(hipMemPoolTrimTo(pool, 0));
    return SPH_OK;
}

int sph_host_malloc(void** ptr, size_t bytes)
{
    SPH_REFUSE_WHILE_CAPTURING();
    SPH_REQUIRE(ptr != nullptr, "ptr is null");
    ::sph::CountAllocation();
    SPH_HIP_TRY(hipHostMalloc(ptr, bytes, hipHostMallocDefault));
    return SPH_OK;
}

int sph_host_free(void* ptr)
{
    SPH_REFUSE_WHILE_CAPTURING();
    SPH_HIP_TRY(hipHostFree(ptr));
    return SPH_OK;
}

int sph_memcpy_h2d(void* dev, const void* host, size_t bytes)
{
    SPH_REFUSE_WHILE_CAPTURING();
    if (bytes == 0)
        return SPH_OK;
    SPH_REQUIRE(dev != nullptr && host != nullptr, "null pointer");
    SPH_STREAM_OR_FAIL(stream);
    SPH_HIP_TRY(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, stream));
    SPH_HIP_TRY(hipStreamSynchronize(stream));
    return SPH_OK;
}

int sph_memcpy_d2h(void* host, const void* dev, size_t bytes)
{
    SPH_REFUSE_WHILE_CAPTURING();
    if (bytes == 0)
        return SPH_OK;
    SPH_REQUIRE(dev != nullptr && host != nullptr, "null pointer");
    SPH_STREAM_OR_FAIL(stream);
    SPH_HIP_TRY(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, stream));
    SPH_HIP_TRY(hipStreamSynchronize(stream));
    return SPH_OK;
}

int sph_memcpy_d2d(void* dst, const void* src, size_t bytes)
{
    SPH_REFUSE_WHILE_CAPTURING();
    if (bytes == 0)
        return SPH_OK;
    SPH_REQUIRE(dst != nullptr && src != nullptr, "null pointer");
    SPH_STREAM_OR_FAIL(stream);
    SPH_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, stream));
    SPH_HIP_TRY(hipStreamSynchronize(stream));
    return SPH_OK;
}

int sph_memcpy_d2d_async(void* dst, const void* src, size_t bytes)
{
    if (bytes == 0)
        return SPH_OK;
    SPH_REQUIRE(dst != nullptr && src != nullptr, "null pointer");
    SPH_STREAM_OR_FAIL(stream);
    SPH_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, stream));
    return SPH_OK;
}

int sph_stream_sync(void)
{
    SPH_REFUSE_WHILE_CAPTURING();
    SPH_STREAM_OR_FAIL(stream);
    SPH_HIP_TRY(hipStreamSynchronize(stream));
    return SPH_OK;
}

int sph_device_sync(void)
{
    SPH_REFUSE_WHILE_CAPTURING();
    SPH_HIP_TRY(hipSetDevice(tlsSlots.device));
    SPH_HIP_TRY(hipDeviceSynchronize());
    return SPH_OK;
}

int sph_stream_wait_stream(void* hipStream)
{
    SPH_REFUSE_WHILE_CAPTURING();
    SPH_STREAM_OR_FAIL(stream);
    hipStream_t other = static_cast<hipStream_t>(hipStream);
    if (other == nullptr || other == stream)
        return SPH_OK;
    hipEvent_t marker = nullptr;
    SPH_HIP_TRY(hipEventCreateWithFlags(&marker, hipEventDisableTiming));
    hipError_t err = hipEventRecord(marker, other);
    if (err == hipSuccess)
        err = hipStreamWaitEvent(stream, marker, 0);
    // the event's resources are released once the wait has been satisfied
    const hipError_t destroyed = hipEventDestroy(marker);
    if (err == hipSuccess)
        err = destroyed;
    if (err != hipSuccess)
        return sph::Fail(SPH_ERR_DEVICE, std::string("sph_stream_wait_stream failed with ") +
                                             hipGetErrorString(err));
    return SPH_OK;
}

int sph_get_stream(void** hipStream)
{
    SPH_REQUIRE(hipStream != nullptr, "hipStream is null");
    SPH_STREAM_OR_FAIL(stream);
    *hipStream = stream;
    return SPH_OK;
}

int sph_set_stream(void* hipStream)
{
    SPH_REFUSE_WHILE_CAPTURING();
    tlsSlots.borrowed[tlsSlots.device] = static_cast<hipStream_t>(hipStream);
    return SPH_OK;
}

int sph_event_create(void** event)
{
    SPH_REQUIRE(event != nullptr, "event is null");
    hipEvent_t ev = nullptr;
    SPH_HIP_TRY(hipEventCreate(&ev));
    *event = ev;
    return SPH_OK;
}

int sph_event_record(void* event)
{
    SPH_REQUIRE(event != nullptr, "event is null");
    SPH_STREAM_OR_FAIL(stream);
    SPH_HIP_TRY(hipEventRecord(static_cast<hipEvent_t>(event), stream));
    return SPH_OK;
}

int sph_event_elapsed_ms(void* start, void* stop, float* ms)
{
    SPH_REFUSE_WHILE_CAPTURING();
    SPH_REQUIRE(start != nullptr && stop != nullptr && ms != nullptr, "null argument");
    SPH_HIP_TRY(hipEventSynchronize(static_cast<hipEvent_t>(stop)));
    SPH_HIP_TRY(hipEventElapsedTime(ms, static_cast<hipEvent_t>(start),
                                    static_cast<hipEvent_t>(stop)));
    return SPH_OK;
}

int sph_event_destroy(void* event)
{
    SPH_REQUIRE(event != nullptr, "event is null");
    SPH_HIP_TRY(hipEventDestroy(static_cast<hipEvent_t>(event)));
    return SPH_OK;
}

int sph_graph_begin_capture(void)
{
    SPH_REQUIRE(!sph::Capturing(), "a capture is already in progress on this thread");
    // resolve everything that queries the device before the stream goes into capture
    (void)sph::ComputeUnits();
    {
        const int rc = sph::ResolveCsrScratch(nullptr);
        if (rc != SPH_OK)
            return rc;
    }
    SPH_STREAM_OR_FAIL(stream);
    {
        // (no other thread hands this stream's block back meanwhile)
        std::lock_guard<std::mutex> lock(gPoolMutex);
        SPH_HIP_TRY(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
    }
    tlsSlots.capturing = stream;
    return SPH_OK;
}

int sph_graph_end_capture(void** graph)
{
    SPH_REQUIRE(graph != nullptr, "graph is null");
    SPH_REQUIRE(sph::Capturing(), "no capture in progress on this thread");
    hipStream_t stream = tlsSlots.capturing;
    tlsSlots.capturing = nullptr;
    *graph = nullptr;
    hipGraph_t recorded = nullptr;
    SPH_HIP_TRY(hipStreamEndCapture(stream, &recorded));
    if (recorded == nullptr)
        return sph::Fail(SPH_ERR_DEVICE, "sph_graph_end_capture - the capture was invalidated");
    hipGraphExec_t exec = nullptr;
    const hipError_t err = hipGraphInstantiate(&exec, recorded, nullptr, nullptr, 0);
    (void)hipGraphDestroy(recorded);
    if (err != hipSuccess)
        return sph::Fail(SPH_ERR_DEVICE, std::string("hipGraphInstantiate failed with ") +
                                             hipGetErrorString(err));
    *graph = exec;
    return SPH_OK;
}

int sph_graph_launch(void* graph)
{
    SPH_REQUIRE(graph != nullptr, "graph is null");
    SPH_REFUSE_WHILE_CAPTURING();
    SPH_STREAM_OR_FAIL(stream);
    SPH_HIP_TRY(hipGraphLaunch(static_cast<hipGraphExec_t>(graph), stream));
    return SPH_OK;
}

int sph_graph_destroy(void* graph)
{
    SPH_REQUIRE(graph != nullptr, "graph is null");
    SPH_HIP_TRY(hipGraphExecDestroy(static_cast<hipGraphExec_t>(graph)));
    return SPH_OK;
}

}  // extern "C"
