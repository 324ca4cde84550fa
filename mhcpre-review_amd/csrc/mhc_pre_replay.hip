// What tells the exchange words of one launch from those of every other: the
// launch tag (see LaunchTag in mhc_pre_internal.h).
//
// Each captured launch gets words of its own in a fixed array of the library's
// device code object, one per workgroup, where every workgroup counts its
// replays.  They are the only memory whose contents the exchange relies on:
// nobody else writes them, all of a launch's words start equal and each replay
// adds one to every one of them, so the workgroups of a replay agree whenever
// they start.
//
// The words belong to the graph: a user object returns them when the graph and
// everything made from it are gone.  A block is handed out again only for the
// same number of workgroups (its words are equal then) and some time after its
// return.  Where none is left, an extra node of the graph sets a block in the
// workspace before each replay instead (2.5 to 3 us).

#include "mhc_pre_internal.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <new>

namespace mhc {
namespace {

constexpr size_t kReplayWords = size_t{1} << 22;  // 16 MiB: 16384 captured launches of 256 workgroups
constexpr int kMaxDevices = 64;
constexpr auto kRest = std::chrono::seconds(2);  // a returned block's replays may still be running

__device__ __align__(256) uint32_t replayWords[kReplayWords];
__device__ uint32_t replayFills;

// The n words of a launch without words of its own: a number that no fill had before.
__global__ __launch_bounds__(256) void fill_words(uint32_t *words, int n)
{
    __shared__ uint32_t value;
    if (threadIdx.x == 0) {
        value = kFilledNumbers |
                __hip_atomic_fetch_add(&replayFills, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    for (int i = (int)threadIdx.x; i < n; i += 256) {
        __hip_atomic_store(words + i, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// The array of one device: words below `used` have been handed out; returned
// blocks wait in `free` under their number of words, oldest first.
struct Pool {
    using Clock = std::chrono::steady_clock;
    struct Block {
        size_t at;
        Clock::time_point since;
    };
    uint32_t *base = nullptr;
    size_t used = 0;
    std::map<int, std::deque<Block>> free;
};
struct Pools {
    std::mutex mu;
    Pool of[kMaxDevices];
};
// (Never destroyed: graphs may outlive static objects.)
Pools &pools()
{
    static Pools *p = new Pools;
    return *p;
}

size_t pool_words()
{
    const char *gate = std::getenv("MHCPRE_TESTING");
    const char *v = gate != nullptr && std::strcmp(gate, "1") == 0 ? std::getenv("MHCPRE_REPLAY_WORDS") : nullptr;
    return v != nullptr ? std::min(kReplayWords, static_cast<size_t>(std::strtoull(v, nullptr, 10))) : kReplayWords;
}

// A block's owner, held by the graph's user object.
struct Lease {
    int device;
    int n;
    size_t at;
};

// Called by the runtime when the last graph that holds the lease is gone.
void give_back(void *p)
{
    Lease *lease = static_cast<Lease *>(p);
    Pools &all = pools();
    {
        std::lock_guard<std::mutex> lock(all.mu);
        try {
            all.of[lease->device].free[lease->n].push_back({lease->at, Pool::Clock::now()});
        } catch (const std::bad_alloc &) {
            // The block stays unused.
        }
    }
    delete lease;
}

// A block of n equal words, or null.
Lease *take(int device, int n)
{
    Lease *lease = new (std::nothrow) Lease{device, n, 0};
    if (lease == nullptr) {
        return nullptr;
    }
    const size_t size = (static_cast<size_t>(n) + 31) / 32 * 32;  // whole 128-byte lines
    const size_t limit = pool_words();
    Pools &all = pools();
    std::lock_guard<std::mutex> lock(all.mu);
    Pool &pool = all.of[device];
    const auto it = pool.free.find(n);
    if (it != pool.free.end() && !it->second.empty() && Pool::Clock::now() - it->second.front().since >= kRest) {
        lease->at = it->second.front().at;
        it->second.pop_front();
        return lease;
    }
    if (pool.used + size <= limit) {
        lease->at = pool.used;
        pool.used += size;
        return lease;
    }
    delete lease;
    return nullptr;
}

}  // namespace

hipError_t replay_words_address(int device, uint32_t **ptr)
{
    if (device < 0 || device >= kMaxDevices) {
        return hipErrorInvalidValue;
    }
    Pools &all = pools();
    {
        std::lock_guard<std::mutex> lock(all.mu);
        *ptr = all.of[device].base;
    }
    if (*ptr != nullptr) {
        return hipSuccess;
    }
    // The caller has made `device` current: its copy of the array.  (Not under
    // the lock, which give_back takes inside calls of the runtime.)
    void *p = nullptr;
    const hipError_t err = hipGetSymbolAddress(&p, HIP_SYMBOL(replayWords));
    if (err != hipSuccess) {
        return err;
    }
    *ptr = static_cast<uint32_t *>(p);
    std::lock_guard<std::mutex> lock(all.mu);
    all.of[device].base = *ptr;
    return hipSuccess;
}

hipError_t make_launch_tag(uint32_t launchId, int device, int grid, void *workspace, hipStream_t stream,
                           LaunchTag &tag)
{
    tag.seed = mix32(launchId & ~kCapturedNumbers);
    tag.words = nullptr;
    if (stream == nullptr) {
        return hipSuccess;  // (the null stream cannot be captured)
    }
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    hipGraph_t graph = nullptr;
    const hipError_t err = hipStreamGetCaptureInfo_v2(stream, &status, nullptr, &graph, nullptr, nullptr);
    if (err != hipSuccess || status != hipStreamCaptureStatusActive) {
        return err;
    }
    static std::atomic<uint32_t> captured{0};
    tag.seed = kCapturedNumbers | ((captured.fetch_add(1u, std::memory_order_relaxed) << kReplayBits) & ~kFilledNumbers);
    uint32_t *base = nullptr;
    if (graph != nullptr && replay_words_address(device, &base) == hipSuccess) {
        if (Lease *lease = take(device, grid)) {
            tag.words = base + lease->at;
            hipUserObject_t object = nullptr;
            if (hipUserObjectCreate(&object, lease, give_back, 1, hipUserObjectNoDestructorSync) != hipSuccess) {
                give_back(lease);
                tag.words = nullptr;
            } else if (hipGraphRetainUserObject(graph, object, 1, hipGraphUserObjectMove) != hipSuccess) {
                (void)hipUserObjectRelease(object, 1);  // (which gives the block back)
                tag.words = nullptr;
            }
        }
    }
    (void)hipGetLastError();
    if (tag.words != nullptr) {
        return hipSuccess;
    }
    tag.words = reinterpret_cast<uint32_t *>(static_cast<char *>(workspace) + kWsReplayOff);
    hipLaunchKernelGGL(fill_words, dim3(1), dim3(256), 0, stream, tag.words, grid);
    return hipGetLastError();
}

}  // namespace mhc
