// host_io.hip — host buffers to the device and back.
//
// A caller's buffers are ordinary pageable memory.  hipMemcpyAsync on such memory goes through the runtime's own staging
// or pins the pages for the transfer: 14 / 22 us for 4 KB in / out, 110 us for 256 KB, 18 GB/s out of the device for
// large results.  Here every transfer goes through pinned memory that the library keeps and is made by a small kernel in the
// caller's stream, so no copy engine has to be synchronised with it.  The host's side of it is a copy by several threads
// (CopyTeam): one moves 28 to 33 GB/s to or from memory that the bus has written or will read, less than the bus itself.  The
// last transfer of a call raises a flag in pinned memory that the host polls: three dependent launches and a poll take 12.6 us
// where the same three and hipStreamSynchronize take 18.
#include <hip/hip_runtime.h>

#include <sched.h>
#include <signal.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "../../include/oxb_hip.h"
#include "host_io.h"
#include "runtime_internal.h"

// 64 workgroups move a large buffer at the rate of the bus; with more of them the fences in front of the flag cost
// more than they gain (1.2 MB out: 34 us with 64 workgroups, 50 with 256).
#define OXB_IO_GRID 64u

// Units of 16 bytes (4, where a buffer lies otherwise), then what is left byte by byte, piece after piece of `piece` bytes.  With
// `flag`: the workgroup that finishes piece c last stores seq + c there once every workgroup's part of it is visible to the host;
// arrived[c] is 0 before and after.  (A workgroup has passed piece c, its store of the flag included, before it counts itself off
// at the next one: the flag only grows.)  One launch for all pieces of a transfer: 19.4 MB out take 387 us, where a launch for
// each piece of 1 MB, the bus idle in between, takes 496 and one without pieces, nothing of it handed over before the end, 362.
// ONE: there is one piece (the smallest calls notice the loop: 0.2 us of 24).
template <typename T, bool ONE>
__global__ __launch_bounds__(256) void io_copy_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, size_t bytes, size_t piece,
                                                       uint32_t* arrived, uint32_t* flag, uint32_t seq) {
    for (uint32_t c = 0; ONE || bytes; c++) {
        const size_t len = ONE || bytes < piece ? bytes : piece, n = len / sizeof(T), step = (size_t)gridDim.x * 256;
        for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += step)
            reinterpret_cast<T*>(dst)[i] = reinterpret_cast<const T*>(src)[i];
        if (blockIdx.x == 0 && threadIdx.x < len % sizeof(T)) dst[n * sizeof(T) + threadIdx.x] = src[n * sizeof(T) + threadIdx.x];
        src += len, dst += len, bytes -= len;
        if (!flag) {
            if (ONE) return;
            continue;
        }
        __threadfence_system();
        __syncthreads();
        if (threadIdx.x == 0) {
            const uint32_t before = __hip_atomic_fetch_add(arrived + c, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
            if (before == gridDim.x - 1) {
                arrived[c] = 0;
                __hip_atomic_store(flag, seq + c, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
            }
        }
        if (ONE) return;
    }
}

namespace oxb {
namespace {

constexpr size_t kChunk = (size_t)1 << 20;      // host copy of one piece while the bus moves the one before
constexpr size_t kStaging = (size_t)32 << 20;   // per direction; larger buffers take turns in it
// Results of up to so many pieces: a launch for each, the first one's copy begins sooner.  Host to host, us, a launch each / one for
// all: 1.3 MB 116 / 123, 2.3 MB 109 / 114, 3.6 MB 140 / 142, 4.6 MB 167 / 166, 6.1 MB 208 / 197, 7.7 MB 249 / 235.
constexpr size_t kFewPieces = 4;
constexpr size_t kPieces = kStaging / kChunk;   // of one launch, at most
constexpr size_t kPoolOut = (size_t)512 << 20;  // result memory handed out at a time
constexpr size_t kPoolKept = (size_t)128 << 20; // ... and kept for reuse
// Calls after which the stream is synchronised all the same, for the runtime to retire its commands (host to host, 1024 x 2048
// GEMV: 17.5 us at the median, 40 to 85 for one call in 256, 17.9 on average).
constexpr uint32_t kSyncEvery = 256;

// The copies of a transfer of more than kShared bytes, shared with up to kHelpers threads of the library's own.  The caller takes
// slices like the helpers and is done when all slices are, so a helper that wakes late costs nothing; a helper looks out for the
// next copy for kLinger and then sleeps.  Used under the library's lock, by one call at a time; io_shutdown ends the threads.
// One thread -> four: 1.3 MB in and out 132 -> 117 us (77 x 4096 GEMM, host to host, call after call), 19 MB out 3.62 -> 3.40 ms (decode of
// 32 sequences), 34 MB in 27.4 -> 26.8 ms (2048-token prefill).  Waking them costs the caller 0.5 to 3 us:
// shared from 64 KB on, a product with 131 KB in and out takes 33.0 us instead of 30.2, with 196 KB 37.3 instead of 37.0; with
// 262 KB it takes 42.8 instead of 43.1, with 328 KB 50.9 instead of 49.4, with 393 KB 48.5 instead of 53.6.
// Helpers that sleep take up to 50 us to come: transfers up to kWake that follow the last one later than kSoon are the caller's alone (a
// decode step of one sequence, 608 KB of logits every 0.8 ms: 8 us less).  A product with so much in and out, 0.3 ms after the last
// one, the caller alone / helpers woken: 0.9 MB 106 / 110 us, 1.0 MB 114 / 117, 1.15 MB 129 / 109 to 127, 1.3 MB 136 / 113 to 132,
// 1.6 MB 153 / 134 to 149, 2.1 MB 170 / 159 to 168, 4.2 MB 277 / 267.
constexpr size_t kShared = (size_t)320 << 10;
constexpr size_t kWake = (size_t)1 << 20;
constexpr auto kSoon = std::chrono::microseconds(100);
constexpr size_t kSlice = (size_t)64 << 10;
constexpr unsigned kHelpers = 3;
constexpr auto kLinger = std::chrono::microseconds(60);
constexpr unsigned kPauses = 4096;  // of the caller's wait for the last slices, some 50 us: then it gives its CPU away each time

// CPUs that this thread may run on.  With a single one nothing is shared: helpers would only take turns with the caller (20 MB in
// pieces of 1 MB: 2.1 ms alone, 4.7 with three helpers on the same CPU).
unsigned cpus_allowed() {
    cpu_set_t set;
    return sched_getaffinity(0, sizeof set, &set) == 0 ? (unsigned)CPU_COUNT(&set) : std::thread::hardware_concurrency();
}

class CopyTeam {
    struct Job {  // what a helper holds on to: a late one sees that no slice is left and lets go
        uint8_t* dst;
        const uint8_t* src;
        size_t bytes;
        std::atomic<size_t> next{0}, done{0};
        Job(uint8_t* d, const uint8_t* s, size_t n) : dst(d), src(s), bytes(n) {}
        void work() {
            for (size_t at; (at = next.fetch_add(kSlice)) < bytes;) {
                const size_t n = std::min(kSlice, bytes - at);
                memcpy(dst + at, src + at, n);
                done.fetch_add(n, std::memory_order_release);
            }
        }
    };
    std::mutex mu;
    std::condition_variable cv;
    std::shared_ptr<Job> job;
    std::atomic<uint64_t> serial{0};
    std::chrono::steady_clock::time_point last{};  // end of the last copy large enough to be shared
    bool stop = false, started = false;
    std::vector<std::thread> threads;

    void run() {
        for (uint64_t seen = 0;;) {
            const auto t0 = std::chrono::steady_clock::now();
            while (serial.load(std::memory_order_acquire) == seen && std::chrono::steady_clock::now() - t0 < kLinger) __builtin_ia32_pause();
            std::shared_ptr<Job> j;
            {
                std::unique_lock<std::mutex> lk(mu);
                cv.wait(lk, [&] { return stop || serial.load() != seen; });
                if (stop) return;
                seen = serial.load();
                j = job;
            }
            if (j) j->work();
        }
    }

public:
    void copy(void* dst, const void* src, size_t bytes, size_t transfer) {  // a piece of a transfer of so many bytes
        if (transfer <= kShared) {
            memcpy(dst, src, bytes);
            return;
        }
        const unsigned cpus = transfer > kWake || std::chrono::steady_clock::now() - last < kSoon ? cpus_allowed() : 1;
        const bool share = cpus > 1;
        if (share && !started) {
            started = true;
            sigset_t all, before;  // the program's signals stay with its own threads
            sigfillset(&all);
            pthread_sigmask(SIG_SETMASK, &all, &before);
            try {
                for (unsigned i = 0; i < kHelpers && i + 1 < cpus; i++) threads.emplace_back([this] { run(); });
            } catch (const std::exception&) {  // no more threads to be had: those there are will do
            }
            pthread_sigmask(SIG_SETMASK, &before, nullptr);
        }
        if (!share || bytes <= kSlice || threads.empty()) {
            memcpy(dst, src, bytes);
            last = std::chrono::steady_clock::now();
            return;
        }
        const std::shared_ptr<Job> j = std::make_shared<Job>((uint8_t*)dst, (const uint8_t*)src, bytes);
        {
            std::lock_guard<std::mutex> lk(mu);
            job = j;
            serial.fetch_add(1, std::memory_order_release);
        }
        cv.notify_all();
        j->work();
        for (unsigned n = 0; j->done.load(std::memory_order_acquire) < bytes; n++) {
            if (n < kPauses) __builtin_ia32_pause();
            else sched_yield();  // (a helper that holds a slice waits for a CPU)
        }
        std::lock_guard<std::mutex> lk(mu);
        job.reset();
        last = std::chrono::steady_clock::now();
    }
    void end() {
        {
            std::lock_guard<std::mutex> lk(mu);
            stop = true;
        }
        cv.notify_all();
        for (std::thread& t : threads) t.join();
        threads.clear();
        stop = started = false;
    }
};
CopyTeam& team = *new CopyTeam;  // (never destroyed: a program may end with its threads asleep)

struct Staging {
    uint8_t *in = nullptr, *out = nullptr;
    size_t in_cap = 0, out_cap = 0, in_used = 0, out_used = 0;
    uint32_t *flag = nullptr, *arrived = nullptr, seq = 0, seq_begin = 0, calls = 0;
    struct Late { void* dst; size_t at, bytes; uint32_t seq; size_t transfer; };
    std::vector<Late> late;  // results that wait in staging for the device
} st;

int staging(uint8_t** p, size_t* cap, size_t want) {  // grows to a power of two up to kStaging; nothing is in flight
    if (want > kStaging) want = kStaging;
    if (*cap >= want) return OXB_HIP_OK;
    size_t n = (size_t)256 << 10;
    while (n < want) n *= 2;
    if (*p) (void)hipHostFree(*p);
    *p = nullptr;
    *cap = 0;
    if (hipHostMalloc((void**)p, n, hipHostMallocCoherent) != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError();
        return fail(OXB_HIP_OUT_OF_MEMORY, "out of host memory: pinned staging of %zu bytes", n);
    }
    *cap = n;
    return OXB_HIP_OK;
}

int ensure_flag() {
    if (st.flag) return OXB_HIP_OK;
    // (the null stream that clears has no order with the stream whose kernels count on it: the clear is waited for)
    if (hipHostMalloc((void**)&st.flag, 64, hipHostMallocCoherent) != hipSuccess || hipMalloc((void**)&st.arrived, kPieces * 4) != hipSuccess ||
        hipMemset(st.arrived, 0, kPieces * 4) != hipSuccess || hipStreamSynchronize(nullptr) != hipSuccess) {
        (void)hipGetLastError();
        if (st.flag) (void)hipHostFree(st.flag);
        if (st.arrived) (void)hipFree(st.arrived);
        st.flag = st.arrived = nullptr;
        return fail(OXB_HIP_OUT_OF_MEMORY, "out of host memory: completion flag");
    }
    *st.flag = st.seq;
    return OXB_HIP_OK;
}

int copy(const void* src, void* dst, size_t bytes, size_t piece, uint32_t* flag, uint32_t seq) {
    const size_t wgs = ((bytes < piece ? bytes : piece) / 16 + 255) / 256;
    const uint32_t grid = wgs < 1 ? 1u : wgs < OXB_IO_GRID ? (uint32_t)wgs : OXB_IO_GRID;
    const uintptr_t at = (uintptr_t)src | (uintptr_t)dst;
    if (at & 3) return fail(OXB_HIP_INVALID_ARGUMENT, "internal error: a buffer of %zu bytes is not aligned to 4", bytes);
    auto run = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, g_rt.stream, (const uint8_t*)src, (uint8_t*)dst, bytes, piece, st.arrived, flag, seq); };
    const bool one = bytes <= piece;
    if (at & 15) one ? run(io_copy_kernel<uint32_t, true>) : run(io_copy_kernel<uint32_t, false>);
    else one ? run(io_copy_kernel<uint4, true>) : run(io_copy_kernel<uint4, false>);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? OXB_HIP_OK : hip_fail(e, "kernel launch failed: io_copy");
}

int sync_all(const char* what) {
    const hipError_t e = hipStreamSynchronize(g_rt.stream);
    return e == hipSuccess ? OXB_HIP_OK : fail(OXB_HIP_SYNC_FAILED, "device synchronization failed: %s: %s", what, hipGetErrorString(e));
}

// Polls for a few milliseconds; a longer wait (or a stream in error, which never raises the flag) is the runtime's.
int wait_for(uint32_t seq, const char* what) {
    const auto t0 = std::chrono::steady_clock::now();
    for (uint32_t n = 1; (int32_t)(__atomic_load_n(st.flag, __ATOMIC_ACQUIRE) - seq) < 0; n++) {
        __builtin_ia32_pause();
        if ((n & 1023u) == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(4)) return sync_all(what);
    }
    return OXB_HIP_OK;
}

// Blocks of pinned memory that are handed out, and those that wait to be: found by size, given back to the system oldest first.
struct Pool {
    struct Kept { uint8_t* p; uint64_t age; };
    std::mutex mu;
    std::map<const uint8_t*, size_t> out;                        // handed out: start -> size
    std::multimap<size_t, Kept> kept;                            // size -> block
    std::map<uint64_t, std::multimap<size_t, Kept>::iterator> by_age;
    uint64_t age = 0;
    size_t out_bytes = 0, kept_bytes = 0;

    uint8_t* take(std::multimap<size_t, Kept>::iterator it) {
        uint8_t* p = it->second.p;
        kept_bytes -= it->first;
        by_age.erase(it->second.age);
        kept.erase(it);
        return p;
    }
    // What has to go so that no more than `limit` bytes are kept; freed by the caller, outside the lock (hipHostFree may
    // wait for the device, and every call asks whether a buffer is pinned).
    void trim(size_t limit, std::vector<uint8_t*>& gone) {
        while (kept_bytes > limit) gone.push_back(take(by_age.begin()->second));
    }
} pool;

void give_back(const std::vector<uint8_t*>& gone) {
    for (uint8_t* p : gone) (void)hipHostFree(p);
}

bool is_pinned(const void* p, size_t bytes) {
    std::lock_guard<std::mutex> lk(pool.mu);
    auto it = pool.out.upper_bound((const uint8_t*)p);
    if (it == pool.out.begin()) return false;
    --it;
    return (const uint8_t*)p + bytes <= it->first + it->second;
}

}  // namespace

int IoCall::begin() {
    int rc = ensure_flag();
    if (rc) return rc;
    open = true;
    st.in_used = st.out_used = 0;
    st.seq_begin = st.seq;
    st.late.clear();
    return OXB_HIP_OK;
}

IoCall::~IoCall() {
    if (open) (void)hipStreamSynchronize(g_rt.stream);
}

int IoCall::upload(void* d_dst, const void* src, size_t bytes) {
    const uint8_t* s = (const uint8_t*)src;
    uint8_t* d = (uint8_t*)d_dst;
    if (((uintptr_t)s & 15) == 0 && is_pinned(s, bytes)) return copy(s, d, bytes, bytes, nullptr, 0);
    int rc;
    if (st.in_used == 0 && (rc = staging(&st.in, &st.in_cap, bytes))) return rc;
    const size_t transfer = bytes;
    while (bytes) {
        const size_t n = bytes < kChunk ? bytes : kChunk;
        if (st.in_used + n > st.in_cap) {  // every piece has been used once: wait for the device to be done with them
            if ((rc = sync_all("input upload"))) return rc;
            st.in_used = 0;
            if ((rc = staging(&st.in, &st.in_cap, bytes))) return rc;
        }
        team.copy(st.in + st.in_used, s, n, transfer);
        if ((rc = copy(st.in + st.in_used, d, n, n, nullptr, 0))) return rc;
        st.in_used += (n + 255) & ~(size_t)255;
        s += n, d += n, bytes -= n;
    }
    return OXB_HIP_OK;
}

int IoCall::download(void* dst, const void* d_src, size_t bytes) {
    if (((uintptr_t)dst & 15) == 0 && is_pinned(dst, bytes)) return copy(d_src, dst, bytes, bytes, st.flag, ++st.seq);
    int rc;
    if (st.out_used == 0 && (rc = staging(&st.out, &st.out_cap, bytes))) return rc;
    const size_t transfer = bytes;
    uint8_t* d = (uint8_t*)dst;
    const uint8_t* s = (const uint8_t*)d_src;
    while (bytes) {
        if (st.out_used + (bytes < kChunk ? bytes : kChunk) > st.out_cap) {  // staging is full of results: hand them over first
            if ((rc = sync_all("output download"))) return rc;
            for (const Staging::Late& l : st.late) team.copy(l.dst, st.out + l.at, l.bytes, l.transfer);
            st.late.clear();
            st.out_used = 0;
            if ((rc = staging(&st.out, &st.out_cap, bytes))) return rc;
        }
        // one launch for all that fits, or for a piece
        const size_t room = st.out_cap - st.out_used, all = transfer <= kFewPieces * kChunk ? std::min(bytes, kChunk) : bytes <= room ? bytes : room / kChunk * kChunk;
        if ((rc = copy(s, st.out + st.out_used, all, kChunk, st.flag, st.seq + 1))) return rc;
        for (size_t at = 0; at < all; at += kChunk) {
            const size_t n = std::min(kChunk, all - at);
            st.late.push_back({d + at, st.out_used, n, ++st.seq, transfer});
            st.out_used += (n + 255) & ~(size_t)255;
        }
        s += all, d += all, bytes -= all;
    }
    return OXB_HIP_OK;
}

int IoCall::finish(const char* what) {
    int rc;
    if (st.seq == st.seq_begin && (rc = sync_all(what))) return rc;  // nothing came back
    for (const Staging::Late& l : st.late) {  // one piece is copied on the host while the next ones cross the bus
        if ((rc = wait_for(l.seq, what))) return rc;
        team.copy(l.dst, st.out + l.at, l.bytes, l.transfer);
    }
    st.late.clear();
    if ((rc = wait_for(st.seq, what))) return rc;
    if (++st.calls % kSyncEvery == 0 && (rc = sync_all(what))) return rc;
    open = false;
    return OXB_HIP_OK;
}

void* pinned_alloc(size_t bytes) {
    if (!bytes) return nullptr;
    const size_t unit = bytes < kChunk ? (size_t)64 << 10 : kChunk, n = (bytes + unit - 1) / unit * unit;
    {
        std::lock_guard<std::mutex> lk(pool.mu);
        // the smallest kept block that is large enough, unless it is more than twice as large
        auto it = pool.kept.lower_bound(n);
        if (it != pool.kept.end() && it->first <= 2 * n && pool.out_bytes + it->first <= kPoolOut) {
            const size_t size = it->first;
            uint8_t* p = pool.take(it);
            pool.out[p] = size;
            pool.out_bytes += size;
            return p;
        }
        if (pool.out_bytes + n > kPoolOut) return nullptr;
        pool.out_bytes += n;  // (room is taken before the lock goes)
    }
    uint8_t* p = nullptr;
    hipError_t e = hipHostMalloc((void**)&p, n, hipHostMallocCoherent);
    if (e != hipSuccess) {  // once more without what is kept
        (void)hipGetLastError();
        std::vector<uint8_t*> gone;
        {
            std::lock_guard<std::mutex> lk(pool.mu);
            pool.trim(0, gone);
        }
        give_back(gone);
        if (!gone.empty() && (e = hipHostMalloc((void**)&p, n, hipHostMallocCoherent)) != hipSuccess) (void)hipGetLastError();
    }
    std::lock_guard<std::mutex> lk(pool.mu);
    if (e == hipSuccess) pool.out[p] = n;
    else p = nullptr, pool.out_bytes -= n;
    return p;
}

bool pinned_free(void* p) {
    std::vector<uint8_t*> gone;
    {
        std::lock_guard<std::mutex> lk(pool.mu);
        auto it = pool.out.find((const uint8_t*)p);
        if (it == pool.out.end()) return false;
        const size_t n = it->second;
        pool.out.erase(it);
        pool.out_bytes -= n;
        pool.by_age[pool.age] = pool.kept.emplace(n, Pool::Kept{(uint8_t*)p, pool.age});
        pool.age++;
        pool.kept_bytes += n;
        pool.trim(kPoolKept, gone);
    }
    give_back(gone);
    return true;
}

void io_shutdown() {  // results that a caller still holds stay
    if (st.in) (void)hipHostFree(st.in);
    if (st.out) (void)hipHostFree(st.out);
    if (st.flag) (void)hipHostFree(st.flag);
    if (st.arrived) (void)hipFree(st.arrived);
    st = Staging();
    team.end();
    std::vector<uint8_t*> gone;
    {
        std::lock_guard<std::mutex> lk(pool.mu);
        pool.trim(0, gone);
    }
    give_back(gone);
}

}  // namespace oxb
