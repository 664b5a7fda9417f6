// Copies between device rows and the caller's ordinary (pageable) memory.
//
// The runtime copies pageable memory through a staging buffer on one thread: 0.94 ms for 16 MB (17 GB/s,
// page-locked 0.30 ms), 7.5 ms for 128 MB, and 31 ms where the destination is fresh (its pages are
// faulted in meanwhile).  Here a few threads move chunks between the caller's memory and page-locked
// slots while the transfers of the next chunks run on the solver's stream.  A pass of 100 steps on 4.2M
// cells with its 134 MB download took 98.6 ms and takes 88.5.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "solver_impl.hpp"

namespace ebb {

namespace {

constexpr size_t MB = size_t(1) << 20;
constexpr unsigned MAX_WORKERS = 8;
constexpr size_t BLOCK_BYTES = MAX_WORKERS * 2 * MB;   // two slots of up to 1 MB per worker
constexpr size_t KEPT_BLOCKS = 2;
// below this the runtime's own staging is as fast: with 1 MB here 24 downloads of 0.2 to 3 MB took a
// 6.81 ms batched pass to 7.08 ms, and a 2 MB state and back took as long either way
constexpr size_t MIN_BYTES = 4 * MB;

}  // namespace

// Page-locked blocks shared by the solvers of the process: a copy leases one, so copies of several
// threads run side by side; at most KEPT_BLOCKS idle ones are kept, and the last solver that used the
// pool frees them.
struct StagePool {
    std::mutex mu;
    std::vector<char*> idle;
    ~StagePool()
    {
        for (char* p : idle) (void)hipHostFree(p);
    }
    char* lease()
    {
        {
            std::lock_guard<std::mutex> g(mu);
            if (!idle.empty()) {
                char* p = idle.back();
                idle.pop_back();
                return p;
            }
        }
        void* p = nullptr;
        if (hipHostMalloc(&p, BLOCK_BYTES, hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        return static_cast<char*>(p);
    }
    void giveBack(char* p)
    {
        {
            std::lock_guard<std::mutex> g(mu);
            if (idle.size() < KEPT_BLOCKS) {
                idle.push_back(p);   // (the capacity is reserved: no exception)
                return;
            }
        }
        (void)hipHostFree(p);
    }
    static std::shared_ptr<StagePool> shared()
    {
        static std::mutex m;
        static std::weak_ptr<StagePool> w;
        std::lock_guard<std::mutex> g(m);
        std::shared_ptr<StagePool> p = w.lock();
        if (!p) {
            p = std::make_shared<StagePool>();
            p->idle.reserve(KEPT_BLOCKS);
            w = p;
        }
        return p;
    }
};

namespace {

// One transfer, shared by its workers: each takes the next chunk, keeps up to two in flight in its own
// two slots, and leaves with both drained.
struct Job {
    char* host;
    char* dev;
    size_t bytes, chunk;
    bool toHost;
    int device;
    hipStream_t stream;
    std::atomic<size_t> next{0};
    std::atomic<int> error{0};

    hipError_t work(char* slots)
    {
        hipEvent_t ev[2] = {nullptr, nullptr};
        size_t at[2] = {bytes, bytes};   // the chunk in each slot (bytes: none)
        hipError_t e = hipSetDevice(device);
        for (int k = 0; k < 2 && e == hipSuccess; k++) e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
        auto finish = [&](int k) {   // waits for slot k's transfer; a download's chunk goes to the caller
            if (at[k] >= bytes) return;
            const hipError_t w = hipEventSynchronize(ev[k]);
            if (e == hipSuccess) e = w;
            if (toHost && w == hipSuccess) std::memcpy(host + at[k], slots + k * MB, std::min(chunk, bytes - at[k]));
            at[k] = bytes;
        };
        for (int k = 0; e == hipSuccess && !error.load(); k ^= 1) {
            finish(k);
            const size_t a = next.fetch_add(chunk);
            if (a >= bytes || e != hipSuccess) break;
            const size_t n = std::min(chunk, bytes - a);
            char* slot = slots + k * MB;
            if (toHost) {
                e = hipMemcpyAsync(slot, dev + a, n, hipMemcpyDeviceToHost, stream);
            } else {
                std::memcpy(slot, host + a, n);
                e = hipMemcpyAsync(dev + a, slot, n, hipMemcpyHostToDevice, stream);
            }
            if (e == hipSuccess) e = hipEventRecord(ev[k], stream);
            // a transfer without its event is waited for before the slots are given up
            if (e == hipSuccess) at[k] = a;
            else (void)hipStreamSynchronize(stream);
        }
        for (int k = 0; k < 2; k++) finish(k);
        for (int k = 0; k < 2; k++)
            if (ev[k]) (void)hipEventDestroy(ev[k]);
        if (e != hipSuccess) error.store(int(e));
        return e;
    }
};

bool pageable(const void* p)
{
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();   // memory that the runtime does not know
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

}  // namespace

hipError_t copyRows(ebb_solver* s, void* host, void* dev, size_t bytes, bool toHost)
{
    auto plain = [&]() {
        const hipError_t e = toHost ? hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s->stream)
                                    : hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s->stream);
        return e;
    };
    if (bytes < MIN_BYTES || !pageable(host)) return plain();
    if (!s->stagePool) s->stagePool = StagePool::shared();
    char* block = s->stagePool->lease();
    if (!block) return plain();
    Job job;
    job.host = static_cast<char*>(host);
    job.dev = static_cast<char*>(dev);
    job.bytes = bytes;
    job.chunk = bytes < 8 * MB ? MB / 2 : MB;
    job.toHost = toHost;
    job.device = s->device;
    job.stream = s->stream;
    // a worker per 4 MB: below that the threads' start costs more than their help
    const size_t cpus = std::max(1u, std::thread::hardware_concurrency() / 2);
    const size_t workers = std::max<size_t>(1, std::min({bytes / (4 * MB), size_t(MAX_WORKERS), cpus}));
    std::vector<std::thread> helpers;
    try {
        helpers.reserve(workers);
        for (size_t w = 1; w < workers; w++) helpers.emplace_back([&job, block, w] { (void)job.work(block + w * 2 * MB); });
    } catch (...) {
        // fewer helpers: the chunks are taken by those that run
    }
    (void)job.work(block);
    for (auto& t : helpers) t.join();
    s->stagePool->giveBack(block);
    return hipError_t(job.error.load());
}

}  // namespace ebb
