// Device context, stream and caching allocator.
// Counterpart of the reference device setup and memory store
// (qgate/simulator/src/CUDADevice.cpp:60-153, MultiDeviceMemoryStore.cpp:164-269), for one GPU:
// no chunking across devices, and no device-wide synchronisation on allocate/free.
#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <thread>
#include <vector>

#include "qg_runtime.hpp"

namespace qg {

void raise_error(const char *fmt, ...) {
    char buf[1024];
    va_list va;
    va_start(va, fmt);
    vsnprintf(buf, sizeof(buf), fmt, va);
    va_end(va);
    throw Error(buf);
}

Runtime &runtime() {
    static Runtime rt;
    return rt;
}

std::string &last_error() {
    thread_local std::string msg;
    return msg;
}

namespace {

// Blocks are kept after free, by size: power-of-two classes up to 1 GiB, larger ones (state vectors
// and pools of 27 and more qubits) in whole 2 MiB. All of them together stay within 8 GiB (another
// allocator of the process, torch's, cannot ask for them back) and 256 MiB, for the tables and
// partial sums beside an 8 GiB state; the block that has been free for longest goes first, so that
// neither size crowds out the other. While large blocks went back to the driver at each free, a
// 28-qubit pool (2 GiB) built again and again, with draws and a marginal, took 67.8 ms a time, 66 of
// them in the driver's allocation and free; kept, 1.64 ms.
constexpr size_t kClassMax = size_t(1) << 30;
constexpr size_t kLargeGrain = size_t(2) << 20;
constexpr size_t kKeptMax = (size_t(8) << 30) + (size_t(256) << 20);

struct Kept {
    void *ptr;
    u64 freed;   // counts up
};
std::map<size_t, std::vector<Kept>> &free_lists() {   // each list oldest first
    static std::map<size_t, std::vector<Kept>> lists;
    return lists;
}
size_t g_cached = 0;
u64 g_frees = 0;

size_t size_class(size_t bytes) {
    if (bytes > kClassMax) return (bytes + kLargeGrain - 1) / kLargeGrain * kLargeGrain;
    size_t c = 256;
    while (c < bytes) c <<= 1;
    return c;
}

// Gives the oldest blocks back until all kept ones are within kKeptMax.
void trim_cache() {
    if (g_cached <= kKeptMax) return;
    QG_HIP(hipStreamSynchronize(runtime().stream));   // queued kernels may still read them
    while (g_cached > kKeptMax) {
        auto oldest = free_lists().end();
        for (auto it = free_lists().begin(); it != free_lists().end(); ++it)
            if (oldest == free_lists().end() || it->second.front().freed < oldest->second.front().freed) oldest = it;
        void *p = oldest->second.front().ptr;
        g_cached -= oldest->first;
        oldest->second.erase(oldest->second.begin());
        if (oldest->second.empty()) free_lists().erase(oldest);
        QG_HIP(hipFree(p));
    }
}

void release_cache() {
    for (auto &kv : free_lists())
        for (const Kept &k : kv.second) hipFree(k.ptr);
    free_lists().clear();
    g_cached = 0;
}

}  // namespace

namespace {
u64 g_piece_items = u64(1) << 30;
}

u64 launch_piece_items() { return g_piece_items; }

namespace {
bool g_register_tiles = true;
}

bool use_register_tiles() { return g_register_tiles; }
void set_register_tiles(bool on) { g_register_tiles = on; }

void set_launch_piece_items(u64 items) {
    QG_REQUIRE(items >= (u64(1) << 12) && items <= (u64(1) << 30) && (items & (items - 1)) == 0,
               "launch piece must be a power of two in [2^12, 2^30]");
    g_piece_items = items;
}

void runtime_init(int device) {
    Runtime &rt = runtime();
    std::lock_guard<std::recursive_mutex> lk(rt.mtx);
    if (rt.initialized) {
        QG_REQUIRE(rt.device == device, "runtime already initialised on device %d", rt.device);
        return;
    }
    int count = 0;
    QG_HIP(hipGetDeviceCount(&count));
    QG_REQUIRE(count > 0, "no HIP device is visible");
    QG_REQUIRE(0 <= device && device < count, "device %d out of range (%d devices)", device, count);
    QG_HIP(hipSetDevice(device));
    hipDeviceProp_t prop;
    QG_HIP(hipGetDeviceProperties(&prop, device));
    rt.device = device;
    rt.n_cus = prop.multiProcessorCount;
    rt.total_mem = prop.totalGlobalMem;
    // default priority stream (non-blocking w.r.t. the legacy null stream)
    QG_HIP(hipStreamCreateWithFlags(&rt.stream, hipStreamNonBlocking));
    QG_HIP(hipMalloc(&rt.d_partials, sizeof(double) * (reduce_grid() + 64)));
    QG_HIP(hipHostMalloc(&rt.h_pinned, sizeof(double) * 64, hipHostMallocDefault));
    rt.initialized = true;
}

namespace {

struct StageBuffers {
    char *buf[2] = {nullptr, nullptr};
    hipEvent_t ev[2] = {nullptr, nullptr};
};

StageBuffers &stage_buffers() {
    static StageBuffers sb;
    return sb;
}

StageBuffers &staging() {
    stream();
    StageBuffers &sb = stage_buffers();
    if (sb.buf[0] == nullptr) {
        for (int b = 0; b < 2; ++b) {
            QG_HIP(hipHostMalloc(reinterpret_cast<void **>(&sb.buf[b]), kStageBytes, hipHostMallocDefault));
            QG_HIP(hipEventCreateWithFlags(&sb.ev[b], hipEventDisableTiming));
        }
    }
    return sb;
}

void release_staging() {
    StageBuffers &sb = stage_buffers();
    for (int b = 0; b < 2; ++b) {
        if (sb.buf[b] != nullptr) hipHostFree(sb.buf[b]);
        if (sb.ev[b] != nullptr) hipEventDestroy(sb.ev[b]);
        sb.buf[b] = nullptr;
        sb.ev[b] = nullptr;
    }
}

char *g_table = nullptr;
bool g_table_busy = false;
double *g_result = nullptr;

void release_tables() {
    if (g_table != nullptr) hipHostFree(g_table);
    if (g_result != nullptr) hipHostFree(g_result);
    g_table = nullptr;
    g_result = nullptr;
    g_table_busy = false;
}

// memcpy split over up to 8 host threads (first touch of fresh pages included)
void parallel_memcpy(char *dst, const char *src, size_t bytes) {
    constexpr size_t kMinPerThread = size_t(4) << 20;
    const unsigned hw = std::max(1u, std::thread::hardware_concurrency());
    const size_t n = std::min<size_t>({8, hw, std::max<size_t>(1, bytes / kMinPerThread)});
    if (n <= 1) {
        std::memcpy(dst, src, bytes);
        return;
    }
    const size_t part = (bytes / n + 4095) & ~size_t(4095);
    std::vector<std::thread> th;
    for (size_t i = 1; i < n; ++i) {
        const size_t off = i * part;
        if (off >= bytes) break;
        const size_t len = std::min(part, bytes - off);
        th.emplace_back([=] { std::memcpy(dst + off, src + off, len); });
    }
    std::memcpy(dst, src, std::min(part, bytes));
    for (std::thread &t : th) t.join();
}

}  // namespace

char *table_buffer() {
    hipStream_t s = stream();
    if (g_table == nullptr)
        QG_HIP(hipHostMalloc(reinterpret_cast<void **>(&g_table), kTableBytes, hipHostMallocDefault));
    if (g_table_busy) QG_HIP(hipStreamSynchronize(s));
    g_table_busy = true;
    return g_table;
}

void table_buffer_done() { g_table_busy = false; }

double *result_buffer() {
    stream();
    if (g_result == nullptr)
        QG_HIP(hipHostMalloc(reinterpret_cast<void **>(&g_result), sizeof(double) * kResultDoubles,
                             hipHostMallocDefault));
    return g_result;
}

HostStager::HostStager() { staging(); }

HostStager::~HostStager() {
    // a stager abandoned by an exception still waits for its copies into the staging buffers
    for (int b = 0; b < 2; ++b)
        if (slot_[b].active) hipEventSynchronize(stage_buffers().ev[b]);
}

void HostStager::drain(int b) {
    StageBuffers &sb = stage_buffers();
    QG_HIP(hipEventSynchronize(sb.ev[b]));
    slot_[b].active = false;
    parallel_memcpy(slot_[b].dst, sb.buf[b], slot_[b].bytes);
}

void HostStager::push(void *dst, const void *src, size_t bytes) {
    QG_REQUIRE(bytes <= kStageBytes, "staged chunk of %zu bytes exceeds the staging buffer", bytes);
    StageBuffers &sb = staging();
    const int b = next_;
    if (slot_[b].active) drain(b);
    QG_HIP(hipMemcpyAsync(sb.buf[b], src, bytes, hipMemcpyDeviceToHost, stream()));
    QG_HIP(hipEventRecord(sb.ev[b], stream()));
    slot_[b].dst = static_cast<char *>(dst);
    slot_[b].bytes = bytes;
    slot_[b].active = true;
    next_ ^= 1;
}

void HostStager::finish() {
    // the older pending chunk sits in buffer next_, the newer one in next_ ^ 1
    for (int k = 0; k < 2; ++k) {
        const int b = next_ ^ k;
        if (slot_[b].active) drain(b);
    }
}

void copy_to_host(void *dst, const void *src, size_t bytes) {
    HostStager st;
    const char *s = static_cast<const char *>(src);
    char *d = static_cast<char *>(dst);
    for (size_t done = 0; done < bytes; done += kStageBytes)
        st.push(d + done, s + done, std::min(kStageBytes, bytes - done));
    st.finish();
}

void runtime_clear() {
    Runtime &rt = runtime();
    std::lock_guard<std::recursive_mutex> lk(rt.mtx);
    if (!rt.initialized) return;
    hipStreamSynchronize(rt.stream);
    release_staging();
    release_tables();
    release_cache();
    hipFree(rt.d_partials);
    hipHostFree(rt.h_pinned);
    hipStreamDestroy(rt.stream);
    rt.d_partials = nullptr;
    rt.h_pinned = nullptr;
    rt.stream = nullptr;
    rt.initialized = false;
}

hipStream_t stream() {
    Runtime &rt = runtime();
    if (!rt.initialized) runtime_init(0);
    return rt.stream;
}

void sync() { QG_HIP(hipStreamSynchronize(stream())); }

void *dev_alloc(size_t bytes) {
    stream();
    if (bytes == 0) bytes = 1;
    Runtime &rt = runtime();
    std::lock_guard<std::recursive_mutex> lk(rt.mtx);
    bytes = size_class(bytes);
    auto it = free_lists().find(bytes);
    if (it != free_lists().end()) {
        void *p = it->second.back().ptr;
        it->second.pop_back();
        if (it->second.empty()) free_lists().erase(it);
        g_cached -= bytes;
        return p;
    }
    void *p = nullptr;
    hipError_t e = hipMalloc(&p, bytes);
    if (e != hipSuccess) {
        // give cached blocks back and retry once
        (void)hipGetLastError();
        sync();
        release_cache();
        e = hipMalloc(&p, bytes);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        raise_error("Out of device memory (requested %zu bytes).", bytes);
    }
    return p;
}

void dev_free(void *ptr, size_t bytes) {
    if (ptr == nullptr) return;
    Runtime &rt = runtime();
    std::lock_guard<std::recursive_mutex> lk(rt.mtx);
    if (bytes == 0) bytes = 1;
    bytes = size_class(bytes);
    if (bytes <= kKeptMax) {
        free_lists()[bytes].push_back(Kept{ptr, ++g_frees});
        g_cached += bytes;
        trim_cache();
        return;
    }
    // the block may still be read by queued kernels: drain the stream first
    QG_HIP(hipStreamSynchronize(rt.stream));
    QG_HIP(hipFree(ptr));
}

void dev_free_quiet(void *ptr, size_t bytes) noexcept {
    try {
        dev_free(ptr, bytes);
    } catch (...) {
    }
}

size_t dev_cached_bytes() { return g_cached; }

}  // namespace qg
