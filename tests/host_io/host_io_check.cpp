// Checks of csrc/host_io.hip against the stand-in runtime of hip/hip_runtime.h; one check per run, named by argv[1].
#include <chrono>
#include <condition_variable>
#include <cstdarg>
#include <cstdio>
#include <deque>
#include <filesystem>
#include <map>
#include <thread>
#include <vector>

#include <sched.h>

#include "../../include/oxb_hip.h"
#include "../../oxibonsai_amd/csrc/host_io.h"
#include "../../oxibonsai_amd/csrc/runtime_internal.h"

thread_local dim3 blockIdx, threadIdx, gridDim;

namespace fake {
size_t syncs = 0, host_mallocs = 0, host_frees = 0, host_bytes = 0, host_bytes_limit = ~(size_t)0;
static std::mutex mu;
static std::condition_variable cv;
static std::deque<std::function<void()>> queue, null_queue;
static bool held = false, busy = false;
static std::map<void*, size_t> host_blocks;

static void device() {
    std::unique_lock<std::mutex> lk(mu);
    for (;;) {
        cv.wait(lk, [] { return !held && !queue.empty(); });
        auto f = std::move(queue.front());
        queue.pop_front();
        busy = true;
        lk.unlock();
        f();
        lk.lock();
        busy = false;
        cv.notify_all();
    }
}
void enqueue(std::function<void()> f) {
    static bool started = (std::thread(device).detach(), true);
    (void)started;
    std::lock_guard<std::mutex> lk(mu);
    queue.push_back(std::move(f));
    cv.notify_all();
}
void hold() {
    std::lock_guard<std::mutex> lk(mu);
    held = true;
}
void release() {
    std::lock_guard<std::mutex> lk(mu);
    held = false;
    cv.notify_all();
}
size_t pending() {
    std::lock_guard<std::mutex> lk(mu);
    return queue.size() + (busy ? 1 : 0);
}
static void drain() {
    std::unique_lock<std::mutex> lk(mu);
    cv.wait(lk, [] { return queue.empty() && !busy; });
}
}  // namespace fake

hipError_t hipStreamSynchronize(hipStream_t stream) {
    if (stream) {
        fake::syncs++;
        fake::drain();
    } else {
        for (auto& f : fake::null_queue) f();
        fake::null_queue.clear();
    }
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
    fake::drain();
    return hipStreamSynchronize(nullptr);
}
hipError_t hipMalloc(void** p, size_t n) {
    *p = malloc(n);
    memset(*p, 0xCD, n);
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    fake::host_mallocs++;
    if (fake::host_bytes + n > fake::host_bytes_limit) return hipErrorOutOfMemory;
    *p = aligned_alloc(4096, (n + 4095) / 4096 * 4096);
    memset(*p, 0xCD, n);
    fake::host_blocks[*p] = n;
    fake::host_bytes += n;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    fake::host_frees++;
    fake::host_bytes -= fake::host_blocks.at(p);
    fake::host_blocks.erase(p);
    free(p);
    return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) {
    fake::null_queue.push_back([=] { memset(p, v, n); });
    return hipSuccess;
}

namespace oxb {
Runtime g_rt;
std::recursive_mutex g_mu;
int fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vfprintf(stderr, fmt, ap);
    fputc('\n', stderr);
    va_end(ap);
    return code;
}
int hip_fail(hipError_t, const char* what) { return fail(OXB_HIP_KERNEL_LAUNCH, "%s", what); }
}  // namespace oxb

using namespace oxb;

#define CHECK(c)                                                        \
    do {                                                                \
        if (!(c)) {                                                     \
            fprintf(stderr, "line %d: %s does not hold\n", __LINE__, #c); \
            fflush(nullptr), _Exit(1);                                                    \
        }                                                               \
    } while (0)

static const size_t MiB = (size_t)1 << 20;

static std::vector<uint8_t> bytes(size_t n, unsigned seed) {
    std::vector<uint8_t> v(n);
    for (size_t i = 0; i < n; i++) v[i] = (uint8_t)((i * 2654435761u + seed) >> 13);
    return v;
}

// There and back through device memory: sizes around a piece, the staging buffer and its multiples, buffers that begin
// off a 16-byte boundary, several buffers in one call.
static void round_trip() {
    const size_t sizes[] = {1, 4, 15, 16, 4096 + 4, 256 * 1024, MiB - 4, MiB, MiB + 20, 5 * MiB + 3, 32 * MiB, 32 * MiB + 8, 71 * MiB + 12};
    std::vector<uint8_t> dev(80 * MiB + 64);
    unsigned seed = 1;
    for (size_t n : sizes)
        for (size_t off : {(size_t)0, (size_t)1, (size_t)8}) {
            std::vector<uint8_t> src = bytes(n + off, seed++), dst(n + off + 4, 0);
            IoCall io;
            CHECK(io.begin() == 0);
            CHECK(io.upload(dev.data(), src.data() + off, n) == 0);
            CHECK(io.download(dst.data() + off, dev.data(), n) == 0);
            CHECK(io.finish("round trip") == 0);
            CHECK(memcmp(dst.data() + off, src.data() + off, n) == 0 && dst[n + off] == 0);
        }
    IoCall io;
    CHECK(io.begin() == 0);
    std::vector<std::vector<uint8_t>> in, out;
    const size_t part[] = {3 * MiB, 20 * MiB, 12, 15 * MiB + 4, 30 * MiB, 4};
    size_t at = 0;
    for (size_t n : part) {
        in.push_back(bytes(n, (unsigned)n)), out.emplace_back(n);
        CHECK(io.upload(dev.data() + at, in.back().data(), n) == 0);
        if (at + (n + 15) / 16 * 16 < 40 * MiB) at += (n + 15) / 16 * 16;
    }
    at = 0;
    CHECK(io.upload(dev.data(), in[4].data(), in[4].size()) == 0);
    for (size_t i = 0; i < out.size(); i++) CHECK(io.download(out[i].data(), dev.data() + 64 * i, out[i].size()) == 0);
    CHECK(io.finish("several buffers") == 0);
    for (size_t i = 0; i < out.size(); i++) {
        const size_t n = std::min(out[i].size(), in[4].size() - 64 * i);
        CHECK(memcmp(out[i].data(), in[4].data() + 64 * i, n) == 0);
    }
}

// A call that ends in an error between its copies and finish: the device is done with the caller's buffers.
static void error_exit() {
    uint8_t* src = (uint8_t*)pinned_alloc(64 * 1024);
    uint8_t* dst = (uint8_t*)pinned_alloc(64 * 1024);
    CHECK(src && dst);
    std::vector<uint8_t> dev(64 * 1024);
    {
        IoCall first;  // (so that nothing below is a first-call clear)
        CHECK(first.begin() == 0 && first.finish("nothing") == 0);
    }
    fake::hold();
    std::thread later([] {
        std::this_thread::sleep_for(std::chrono::milliseconds(50));
        fake::release();
    });
    {
        IoCall io;
        CHECK(io.begin() == 0);
        CHECK(io.upload(dev.data(), src, 64 * 1024) == 0);
        CHECK(io.download(dst, dev.data(), 64 * 1024) == 0);
    }
    CHECK(fake::pending() == 0);
    later.join();
}

// The counter behind the completion flag is clear before the first kernel counts on it, whatever the null stream is doing:
// the flag comes up by itself, from the first call on.
static void first_call() {
    std::vector<uint8_t> dev(4096), dst(4096);
    for (int i = 0; i < 8; i++) {
        IoCall io;
        CHECK(io.begin() == 0);
        const size_t before = fake::syncs;
        CHECK(io.upload(dev.data(), dst.data(), 4096) == 0);
        CHECK(io.download(dst.data(), dev.data(), 4096) == 0);
        CHECK(io.finish("a call") == 0);
        CHECK(fake::syncs == before);
        if (i == 3) (void)hipDeviceSynchronize();
    }
}

// Blocks of sizes that come again or lie close by are reused, however much else is kept; what is kept stays within 128 MiB,
// what is handed out within 512 MiB, and where memory runs out what is kept goes first.
static void pool_of_results() {
    std::vector<void*> all;
    for (int i = 0; i < 128; i++) all.push_back(pinned_alloc(MiB));
    for (void* p : all) CHECK(p && pinned_free(p));
    CHECK(fake::host_mallocs == 128 && fake::host_frees == 0 && fake::host_bytes == 128 * MiB);
    // another size while the pool is full: one new block, not one for every result
    for (int i = 0; i < 100; i++) {
        void* p = pinned_alloc(3 * MiB + 1);
        CHECK(p && pinned_free(p));
        CHECK(fake::host_bytes <= 128 * MiB);
    }
    CHECK(fake::host_mallocs == 129);
    // ragged sizes: every result fits a block that is there
    for (size_t n = 600 * 1024; n < MiB; n += 5 * 1024) {
        void* p = pinned_alloc(n);
        CHECK(p && pinned_free(p));
    }
    CHECK(fake::host_mallocs == 129);
    // sizes that change for good: the old ones make room
    all.clear();
    for (int i = 0; i < 16; i++) all.push_back(pinned_alloc(8 * MiB));
    for (void* p : all) CHECK(p && pinned_free(p));
    CHECK(fake::host_bytes == 128 * MiB && fake::host_mallocs == 129 + 16);
    for (int i = 0; i < 16; i++) all[i] = pinned_alloc(8 * MiB);
    CHECK(fake::host_mallocs == 129 + 16);
    for (void* p : all) CHECK(pinned_free(p));
    CHECK(!pinned_free(all[0]) && !pinned_free(&all));
    // the bound on what is handed out
    all.clear();
    for (int i = 0; i < 8; i++) all.push_back(pinned_alloc(64 * MiB));
    for (void* p : all) CHECK(p);
    CHECK(!pinned_alloc(1) && !pinned_alloc(0));
    CHECK(pinned_free(all[7]));
    CHECK((all[7] = pinned_alloc(1)) != nullptr);
    for (void* p : all) CHECK(pinned_free(p));
    CHECK(fake::host_bytes <= 128 * MiB);
    // out of memory: what is kept is given up for the request
    fake::host_bytes_limit = 100 * MiB;
    void* p = pinned_alloc(90 * MiB);
    CHECK(p && fake::host_bytes == 90 * MiB);
    CHECK(!pinned_alloc(20 * MiB) && pinned_free(p));
    CHECK((p = pinned_alloc(20 * MiB)) && pinned_free(p));
    io_shutdown();
    CHECK(fake::host_bytes == 0);
}

static size_t threads() {
    size_t n = 0;
    for (const auto& e : std::filesystem::directory_iterator("/proc/self/task")) (void)e, n++;
    return n;
}

static void there_and_back(size_t n, unsigned seed) {
    static std::vector<uint8_t> dev(32 * MiB);
    std::vector<uint8_t> src = bytes(n, seed), dst(n, 0);
    IoCall io;
    CHECK(io.begin() == 0);
    CHECK(io.upload(dev.data(), src.data(), n) == 0 && io.download(dst.data(), dev.data(), n) == 0 && io.finish("there and back") == 0);
    CHECK(src == dst);
}

// A caller that may run on one CPU gets no helpers; on two it gets one; and with all threads on one CPU while helpers are there
// the copies end.
static void few_cpus() {
    cpu_set_t all, some;
    CHECK(sched_getaffinity(0, sizeof all, &all) == 0);
    std::vector<int> cpus;
    for (int i = 0; i < CPU_SETSIZE; i++)
        if (CPU_ISSET(i, &all)) cpus.push_back(i);
    there_and_back(64, 1);  // (the stand-in's device has its thread)
    const size_t before = threads();
    CPU_ZERO(&some);
    CPU_SET(cpus[0], &some);
    CHECK(sched_setaffinity(0, sizeof some, &some) == 0);
    for (unsigned i = 0; i < 4; i++) there_and_back(20 * MiB + 4, i);
    CHECK(threads() == before);
    if (cpus.size() > 1) {
        CPU_SET(cpus[1], &some);
        CHECK(sched_setaffinity(0, sizeof some, &some) == 0);
        for (unsigned i = 0; i < 4; i++) there_and_back(20 * MiB + 4, i);
        CHECK(threads() == before + 1);
        CPU_CLR(cpus[1], &some);
        for (const auto& e : std::filesystem::directory_iterator("/proc/self/task"))
            CHECK(sched_setaffinity(std::stoi(e.path().filename()), sizeof some, &some) == 0);
        for (unsigned i = 0; i < 4; i++) there_and_back(20 * MiB + 4, i);
    }
    io_shutdown();
    for (int i = 0; i < 1000 && threads() != before; i++) std::this_thread::sleep_for(std::chrono::milliseconds(1));  // (the system's list lags behind)
    CHECK(threads() == before);
}

int main(int argc, char** argv) {
    g_rt.stream = g_rt.own_stream = (hipStream_t)&g_rt;
    const struct { const char* name; void (*run)(); } checks[] = {{"round_trip", round_trip}, {"error_exit", error_exit}, {"first_call", first_call}, {"pool_of_results", pool_of_results}, {"few_cpus", few_cpus}};
    for (const auto& c : checks)
        if (argc == 2 && !strcmp(argv[1], c.name)) {
            c.run();
            fflush(nullptr);
            _Exit(0);
        }
    return 2;
}
