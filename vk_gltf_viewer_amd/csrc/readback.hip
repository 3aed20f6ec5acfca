// Device to host readback.
//
// The runtime's copy into pageable memory goes through staging of its own, a
// copy and a memcpy in turn: 17 GB/s.  Here one kernel writes the data to a
// pinned stage in pieces of kPiece bytes, in order, and raises a flag in it
// after each, and the host copies a piece out as soon as its flag is up, while
// the next ones cross the bus.  The kernel is kept to kBlocks blocks, so that
// the pieces finish one after another (all of 4 MB at once finished together:
// 93 us and then 100 us of memcpy; 16 blocks 134 us in all, 211 -> 115 us for
// 3.7 MB against the runtime).  No call into the runtime between the pieces:
// an async copy and an event per megabyte cost as much as they hid.
// The stage is two halves, a kernel each; a half is launched again when the
// host has emptied it, so that a read of any size keeps the bus busy.
//
// The kernel's launch and its pieces cost some 7 us more than a small plain copy
// does on an idle stream: 64 KB 20 us against 12, 512 KB 36 against 30, equal at
// 896 KB (47), 1 MB 50 against 61.  Behind a frame that is still running the
// launch is hidden: a 480x270 frame with its 506 KB of colour 94 us against 96,
// 560x400 with 875 KB 104 against 110, equal up to 300 KB.  So a read of
// kReadStaged bytes is staged while the stream is busy, one of kReadStagedIdle
// always.  A plain copy waits for the stream first: queued behind a frame it takes
// the runtime 15 us more (a 96x64 frame with its colour 95 us, not 80).
#include <algorithm>
#include <array>
#include <atomic>
#include <cstring>
#include <mutex>

#include "internal.hpp"

namespace vkgv {
namespace {

constexpr size_t kPiece = 16u << 10;
constexpr uint32_t kHalfPieces = 128;                       // 2 MB a half
constexpr size_t kHalfBytes = kPiece * kHalfPieces;
constexpr uint32_t kBlocks = 16, kThreads = 256;

// Pieces blockIdx.x, + gridDim.x, ...: 16-byte words, then the last bytes (a
// multiple of 4) as words.  Every thread makes its stores visible to the host
// before the piece's flag is stored.
__global__ __launch_bounds__(kThreads) void stage_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ stage,
                                                         size_t bytes, uint32_t* __restrict__ flags, uint32_t epoch)
{
    for (size_t p = blockIdx.x; p * kPiece < bytes; p += gridDim.x) {
        const size_t first = p * kPiece, n = min(kPiece, bytes - first), n16 = n / 16;
        const uint4* s = reinterpret_cast<const uint4*>(src + first);
        uint4* d = reinterpret_cast<uint4*>(stage + first);
#pragma unroll 4
        for (size_t k = threadIdx.x; k < n16; k += kThreads) d[k] = s[k];
        const size_t rest = n16 * 4 + threadIdx.x;
        if (rest < n / 4)
            reinterpret_cast<uint32_t*>(stage + first)[rest] = reinterpret_cast<const uint32_t*>(src + first)[rest];
        __threadfence_system();
        __syncthreads();
        if (threadIdx.x == 0) __hip_atomic_store(&flags[p], epoch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// A pinned stage: the two halves' bytes, then their flags.  The host reads both
// while the kernel that stores them runs, so the memory is asked for as
// coherent: without the flag its kind is left to the environment, and other
// memory is only promised to be up to date once the kernel has ended.
struct Stage {
    uint8_t* bytes = nullptr;
    uint32_t* flags = nullptr;
    uint32_t epoch = 0;
};

// Idle stages, shared by the contexts of the process (any device: the memory
// is portable).  At most kIdle are kept, and none once the last context is
// gone; a readback owns the stage it took until it returns.
constexpr size_t kIdle = 2;
std::mutex g_mutex;
std::array<Stage, kIdle> g_idle;   // the first g_idle_count
size_t g_idle_count = 0;
uint32_t g_users = 0;

bool take_stage(Stage& s)
{
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        if (g_idle_count) {
            s = g_idle[--g_idle_count];
            return true;
        }
    }
    void* p = nullptr;
    const size_t flag_bytes = sizeof(uint32_t) * 2 * kHalfPieces;
    if (hipHostMalloc(&p, 2 * kHalfBytes + flag_bytes, hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    s.bytes = static_cast<uint8_t*>(p);
    s.flags = reinterpret_cast<uint32_t*>(s.bytes + 2 * kHalfBytes);
    std::memset(s.flags, 0, flag_bytes);
    return true;
}

void give_stage(const Stage& s)
{
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        if (g_users && g_idle_count < kIdle) {
            g_idle[g_idle_count++] = s;
            return;
        }
    }
    (void)hipHostFree(s.bytes);
}

// Waits until the stage's piece is there.  The stream is asked now and
// then, so that a failed kernel ends the wait; one that has finished has
// stored its flags.
hipError_t wait_flag(const uint32_t* flag, uint32_t epoch, hipStream_t st)
{
    const std::atomic<uint32_t>& f = *reinterpret_cast<const std::atomic<uint32_t>*>(flag);
    for (uint32_t spin = 1;; ++spin) {
        if (f.load(std::memory_order_acquire) == epoch) return hipSuccess;
        __builtin_ia32_pause();
        if (spin % 4096u == 0u) {
            const hipError_t e = hipStreamQuery(st);
            if (e == hipSuccess) return hipSuccess;
            if (e != hipErrorNotReady) return e;
            (void)hipGetLastError();
        }
    }
}

bool busy(hipStream_t st)
{
    if (hipStreamQuery(st) != hipErrorNotReady) return false;   // an error is reported by the copy
    (void)hipGetLastError();
    return true;
}

bool pageable(const void* p)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();   // memory the runtime does not know
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

} // namespace

void read_back_user(bool joins)
{
    std::array<Stage, kIdle> gone;
    size_t n = 0;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        g_users += joins ? 1u : ~0u;
        if (g_users == 0) {
            gone = g_idle;
            n = g_idle_count;
            g_idle_count = 0;
        }
    }
    for (size_t k = 0; k < n; ++k) (void)hipHostFree(gone[k].bytes);
}

hipError_t read_back(void* dst, const void* src, size_t bytes, hipStream_t st)
{
    Stage s;
    const bool words = bytes % 4 == 0 && reinterpret_cast<uintptr_t>(src) % 16 == 0;
    const bool large = bytes >= kReadStagedIdle || (bytes >= kReadStaged && busy(st));
    if (!large || !words || !pageable(dst) || !take_stage(s)) {
        hipError_t e = hipStreamSynchronize(st);
        if (e == hipSuccess) e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
        return e == hipSuccess ? hipStreamSynchronize(st) : e;
    }
    const size_t n = (bytes + kHalfBytes - 1) / kHalfBytes;   // halves to go through
    const uint32_t epoch0 = s.epoch;
    size_t sent = 0;
    hipError_t e = hipSuccess;
    for (size_t k = 0; k < n && e == hipSuccess; ++k) {
        for (; sent < n && sent < k + 2 && e == hipSuccess; ++sent) {
            const size_t first = sent * kHalfBytes, m = std::min(kHalfBytes, bytes - first);
            stage_kernel<<<(uint32_t)std::min<size_t>(kBlocks, (m + kPiece - 1) / kPiece), kThreads, 0, st>>>(
                static_cast<const uint8_t*>(src) + first, s.bytes + (sent & 1) * kHalfBytes, m,
                s.flags + (sent & 1) * kHalfPieces, ++s.epoch);
            e = hipGetLastError();
        }
        const size_t first = k * kHalfBytes, m = std::min(kHalfBytes, bytes - first);
        for (size_t b = 0; b * kPiece < m && e == hipSuccess; ++b) {
            e = wait_flag(s.flags + (k & 1) * kHalfPieces + b, epoch0 + (uint32_t)k + 1u, st);
            if (e == hipSuccess)
                std::memcpy(static_cast<uint8_t*>(dst) + first + b * kPiece,
                            s.bytes + (k & 1) * kHalfBytes + b * kPiece, std::min(kPiece, m - b * kPiece));
        }
    }
    // the kernels have stored their last flags; a stage that goes back is no longer written
    const hipError_t end = hipStreamSynchronize(st);
    give_stage(s);
    return e != hipSuccess ? e : end;
}

} // namespace vkgv
