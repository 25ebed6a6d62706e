// Status reporting and the per-stream scratch arena behind every entry point.
#include "common.hpp"

#include <map>
#include <mutex>
#include <utility>
#include <vector>

namespace cgptx {
namespace {

thread_local std::string g_last_error;

struct Arena {
    void* data = nullptr;
    std::size_t bytes = 0;
    std::uint64_t generation = 0;  // value of g_generation when this block was allocated
    unsigned int* tickets = nullptr;
    bool recorded = false;       // a caller's graph may hold this block's address
    std::vector<void*> retired;  // earlier blocks of which that was so
};
thread_local int g_watches = 0;  // see ScratchWatch

std::mutex g_arena_mutex;
std::map<std::pair<int, hipStream_t>, Arena> g_arenas;
std::uint64_t g_generation = 0;  // bumped by every allocation; a released arena reads as generation 0

}  // namespace

int fail(int code, const std::string& message) {
    g_last_error = message;
    return code;
}

void clear_error() { g_last_error.clear(); }

int check_hip(hipError_t error, const char* what) {
    if (error == hipSuccess) return CGPTX_OK;
    return fail(CGPTX_RUNTIME, std::string(what) + ": " + hipGetErrorString(error));
}

ScratchWatch::ScratchWatch() { ++g_watches; }
ScratchWatch::~ScratchWatch() { --g_watches; }

// Grows the stream's arena to `bytes` where that is possible. *data, *held: the arena as it then is. *capturing, *allocation: what
// was in the way if it holds less.
static int grow_arena(hipStream_t stream, std::size_t bytes, void** data, std::size_t* held, bool* capturing, hipError_t* allocation) {
    int device = 0;
    CGPTX_HIP(hipGetDevice(&device));
    std::lock_guard<std::mutex> lock(g_arena_mutex);
    Arena& arena = g_arenas[{device, stream}];
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (stream != nullptr && (arena.bytes < bytes || !arena.recorded)) CGPTX_HIP(hipStreamIsCapturing(stream, &capture));
    *capturing = capture != hipStreamCaptureStatusNone;
    if (*capturing && g_watches == 0) arena.recorded = true;
    if (arena.bytes < bytes) {
        // Round up so that small variations in problem size do not reallocate.
        const std::size_t rounded = (bytes + (std::size_t{1} << 20) - 1) & ~((std::size_t{1} << 20) - 1);
        void* fresh = nullptr;
        if (!*capturing) *allocation = hipMalloc(&fresh, rounded);
        if (*allocation != hipSuccess) (void)hipGetLastError();  // reported from here, not by the next launch
        if (fresh != nullptr) {
            if (arena.data != nullptr) {
                // hipFree waits for outstanding work that may still read the old block. One that a recorded call of the caller's works
                // in stays until cgptx_release_scratch: its graph may be replayed at any time.
                if (arena.recorded) arena.retired.push_back(arena.data);
                else CGPTX_HIP(hipFree(arena.data));
            }
            arena.data = fresh;
            arena.bytes = rounded;
            arena.recorded = false;
            arena.generation = ++g_generation;
        }
    }
    *data = arena.data;
    *held = arena.bytes;
    return CGPTX_OK;
}

int scratch(hipStream_t stream, std::size_t bytes, void** out) {
    std::size_t held = 0;
    bool capturing = false;
    hipError_t allocation = hipSuccess;
    if (int s = grow_arena(stream, bytes, out, &held, &capturing, &allocation)) return s;
    if (held < bytes && capturing)
        return fail(CGPTX_CAPTURE_ALLOC,
                    "scratch arena would have to grow during stream capture; run the op once eagerly first");
    CGPTX_HIP(allocation);
    return CGPTX_OK;
}

int scratch_up_to(hipStream_t stream, std::size_t bytes, void** out, std::size_t* held) {
    bool capturing = false;
    hipError_t allocation = hipSuccess;
    return grow_arena(stream, bytes, out, held, &capturing, &allocation);
}

unsigned int* tickets(hipStream_t stream) {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return nullptr;
    std::lock_guard<std::mutex> lock(g_arena_mutex);
    Arena& arena = g_arenas[{device, stream}];
    if (arena.tickets != nullptr) return arena.tickets;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (stream != nullptr && hipStreamIsCapturing(stream, &capture) != hipSuccess) capture = hipStreamCaptureStatusActive;
    void* fresh = nullptr;
    constexpr std::size_t bytes = kTickets * sizeof(unsigned int);
    if (capture != hipStreamCaptureStatusNone || hipMalloc(&fresh, bytes) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    if (hipMemsetAsync(fresh, 0, bytes, stream) != hipSuccess) {
        (void)hipGetLastError();
        (void)hipFree(fresh);
        return nullptr;
    }
    arena.tickets = static_cast<unsigned int*>(fresh);
    return arena.tickets;
}

std::uint64_t scratch_generation(hipStream_t stream) {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return 0;
    std::lock_guard<std::mutex> lock(g_arena_mutex);
    const auto it = g_arenas.find({device, stream});
    return it == g_arenas.end() ? 0 : it->second.generation;
}

int compute_units() {
    static int cached = [] {
        int device = 0;
        int count = 0;
        if (hipGetDevice(&device) != hipSuccess ||
            hipDeviceGetAttribute(&count, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || count <= 0) {
            count = 256;
        }
        return count;
    }();
    return cached;
}

}  // namespace cgptx

extern "C" const char* cgptx_last_error(void) { return cgptx::g_last_error.c_str(); }

extern "C" const char* cgptx_version(void) { return "cgptx 0.1 (gfx950)"; }

extern "C" size_t cgptx_scratch_bytes(cgptx_stream stream) {
    using namespace cgptx;
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return 0;
    std::lock_guard<std::mutex> lock(g_arena_mutex);
    const auto it = g_arenas.find({device, static_cast<hipStream_t>(stream)});
    return it == g_arenas.end() ? 0 : it->second.bytes;
}

extern "C" int cgptx_release_scratch(void) {
    using namespace cgptx;
    int device = 0;
    CGPTX_HIP(hipGetDevice(&device));
    CGPTX_HIP(hipDeviceSynchronize());
    std::lock_guard<std::mutex> lock(g_arena_mutex);
    for (auto it = g_arenas.begin(); it != g_arenas.end();) {
        if (it->first.first == device) {
            if (it->second.data != nullptr) CGPTX_HIP(hipFree(it->second.data));
            if (it->second.tickets != nullptr) CGPTX_HIP(hipFree(it->second.tickets));
            for (void* block : it->second.retired) CGPTX_HIP(hipFree(block));
            it = g_arenas.erase(it);
        } else {
            ++it;
        }
    }
    return CGPTX_OK;
}
