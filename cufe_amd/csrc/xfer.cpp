// xfer.cpp -- the library's device blocks and its large copies to and from
// pageable host memory.
//
// Device blocks.  The entry points hold their buffers for one call.  hipMalloc
// and hipFree of the hundreds of MB a model or a row store needs cost 0.05 to
// 0.4 ms each, and calls that follow one another wait for the driver to give
// the freed memory out again (a 2,000-SV model rebuilt in a loop: 2.2 to 9.9 ms
// a pass, 1.4 with the blocks kept).  Blocks are therefore kept when a DevBuf
// lets go of them and handed to the next one they fit, up to kPoolBytes per
// process; beyond that those released longest ago are freed (a process whose
// sizes change would otherwise sit on blocks it no longer asks for), and
// everything kept is freed when an allocation fails.  A block of up to kClassMax
// bytes is rounded up by an eighth at most, so that calls of similar sizes share
// it (8 MiB at most lost); a larger one has its own size, and is kept for
// requests down to eight ninths of it.  Buffers that stay and are counted against
// a budget or fill the card (models, row stores, a server's slots) are exact:
// their own size, new or kept.  hipFree also waited for the device, so a
// block could be let go of with work in flight (an error return between
// launches); here the device is waited for before a block released since the
// last wait is handed out again.
//
// Copies.  A copy to pageable memory runs at 17 GB/s through the runtime, and
// one from it at 29 to 39; one core copying and taking the page faults is the
// limit, not the link (57 GB/s).  Large copies go through pinned chunks
// instead, a few threads each copying a chunk to or from the caller while the
// others' chunks cross the link: the reference's 38.6 MB keys 2.2 -> 0.95 ms out,
// 1.35 -> 0.9 in (a whole key generation).  Waking the threads, filling and
// draining their chunks costs a small copy some 0.06 ms, so it gains less: out
// 16.8 MB 0.97 -> 0.47 ms, 8.4 MB 0.49 -> 0.31, 6.3 MB 0.37 -> 0.27, 4.2 MB level,
// and from kStageDown bytes on they take them.  In, a key generation over 4.2,
// 6.3, 8.4, 12.6 and 16.8 MB takes 181, 228, 293, 395 and 510 us with the runtime's
// copy where the caches hold the source, 226, 295, 380, 522 and 678 where they do
// not, and 245, 270, 305, 400 and 465 (280, 312, 357, 434 and 537) with the threads:
// from kStageUp on, except beside a stream's work, where the runtime's copy
// would wait for it.  Six threads and eight give the same, more than eight are
// slower; chunks of 1 MiB load at 30 GB/s.
#include <hip/hip_runtime.h>
#include <sched.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "runtime.h"

namespace ipfe {

// ---------------------------------------------------------------------------
// Device blocks
// ---------------------------------------------------------------------------
namespace {

constexpr size_t kPoolBytes = (size_t)4 << 30;  // kept at most; larger blocks are never kept
constexpr size_t kClassMax = (size_t)64 << 20;  // rounded up to here

struct Block {
    void *p;
    uint64_t released;  // release number
};

struct Pool {
    std::mutex mu;
    std::map<std::pair<int, size_t>, std::vector<Block>> free;  // by device and size; none empty
    std::map<void *, std::pair<int, size_t>> live;
    size_t kept = 0;
    uint64_t releases = 0;
    std::map<int, uint64_t> waited;  // a device's blocks released up to here are idle
};

// Never destroyed: the process's end gives the blocks back, in no set order
// with the HIP runtime's own.
Pool &pool()
{
    static Pool *p = new Pool();
    return *p;
}

// A request's own size, and the size a new block for it has.
size_t own_size(size_t bytes) { return (bytes + 511) / 512 * 512; }
size_t block_size(size_t bytes, bool exact)
{
    if (exact || bytes > kClassMax) return own_size(bytes);
    size_t step = 512;  // of the sizes from 8 to 16 steps
    while (step * 16 <= bytes) step *= 2;
    return (bytes + step - 1) / step * step;
}

// Frees what is kept (mu held).
void drop_all(Pool &pl)
{
    for (auto &f : pl.free)
        for (const Block &b : f.second) (void)hipFree(b.p);
    pl.free.clear();
    pl.kept = 0;
}

// Frees the block kept longest (mu held, something is kept).
void drop_oldest(Pool &pl)
{
    auto old = pl.free.end();
    for (auto it = pl.free.begin(); it != pl.free.end(); ++it)
        if (old == pl.free.end() || it->second.front().released < old->second.front().released) old = it;
    (void)hipFree(old->second.front().p);
    pl.kept -= old->first.second;
    old->second.erase(old->second.begin());
    if (old->second.empty()) pl.free.erase(old);
}

}  // namespace

static int take_block(void **out, size_t bytes, bool exact)
{
    Pool &pl = pool();
    int dev = 0;
    HIP_OK(hipGetDevice(&dev));
    std::pair<int, size_t> key(dev, block_size(bytes, exact));
    std::lock_guard<std::mutex> lk(pl.mu);
    // the smallest kept block that holds it
    auto it = pl.free.lower_bound(key);
    if (it != pl.free.end() && it->first.first == dev &&
        it->first.second <= (exact ? key.second : key.second + key.second / 8)) {
        // the block released first is the likeliest to be idle already
        const Block b = it->second.front();
        uint64_t &waited = pl.waited[dev];
        if (b.released <= waited || hipDeviceSynchronize() == hipSuccess) {
            if (b.released > waited) waited = pl.releases;
            pl.live[b.p] = it->first;
            pl.kept -= it->first.second;
            it->second.erase(it->second.begin());
            if (it->second.empty()) pl.free.erase(it);
            *out = b.p;
            return 0;
        }
        (void)hipGetLastError();
    }
    hipError_t e = hipMalloc(out, key.second);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        drop_all(pl);
        key.second = own_size(bytes);
        e = hipMalloc(out, key.second);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        *out = nullptr;
        ipfe_set_error("hipMalloc of %zu bytes failed: %s", bytes, hipGetErrorString(e));
        return -1;
    }
    try {
        pl.live[*out] = key;
    } catch (...) {
        (void)hipFree(*out);
        *out = nullptr;
        throw;
    }
    return 0;
}

// Callers are entry points of the C ABI and destructors: host memory that runs
// out for the pool's own records is an error like the device's.
int dev_alloc(void **out, size_t bytes, bool exact)
{
    *out = nullptr;
    try {
        return take_block(out, bytes, exact);
    } catch (...) {
        ipfe_set_error("no host memory to record a block of %zu bytes", bytes);
        return -1;
    }
}

void dev_trim()
{
    Pool &pl = pool();
    std::lock_guard<std::mutex> lk(pl.mu);
    drop_all(pl);
}

void dev_free(void *p)
{
    if (!p) return;
    Pool &pl = pool();
    std::lock_guard<std::mutex> lk(pl.mu);
    auto it = pl.live.find(p);
    if (it == pl.live.end()) return;
    const std::pair<int, size_t> key = it->second;
    pl.live.erase(it);
    if (key.second > kPoolBytes) {
        (void)hipFree(p);
        return;
    }
    while (pl.kept + key.second > kPoolBytes) drop_oldest(pl);
    try {
        auto &kept = pl.free[key];
        try {
            kept.push_back(Block{p, pl.releases + 1});
        } catch (...) {
            if (kept.empty()) pl.free.erase(key);
            throw;
        }
        ++pl.releases;
        pl.kept += key.second;
    } catch (...) {
        (void)hipFree(p);
    }
}

// ---------------------------------------------------------------------------
// Copies
// ---------------------------------------------------------------------------
namespace {

constexpr size_t kStageDown = (size_t)4 << 20, kStageUp = (size_t)8 << 20;
constexpr size_t kChunk = (size_t)2 << 20;
constexpr int kMaxCopyThreads = 8;

struct Lane {  // one copy thread's stream and pinned chunks
    hipStream_t st = nullptr;
    hipEvent_t ev[2] = {};
    uint8_t *slot[2] = {};
};

class Copier {
public:
    // nullptr where the threads, their pinned or other memory cannot be had
    static Copier *get(int dev)
    {
        static std::mutex mu;
        static std::map<int, Copier *> &all = *new std::map<int, Copier *>();  // never destroyed, as the pool
        std::lock_guard<std::mutex> lk(mu);
        auto it = all.find(dev);
        if (it == all.end()) {
            it = all.emplace(dev, nullptr).first;
            Copier *c = new Copier(dev);
            if (c->ok) it->second = c;
            else delete c;
        }
        return it->second;
    }

    // Copies, after what st holds already unless beside is set; false when
    // another copy holds the threads (nothing done).
    bool run(uint8_t *dst, const uint8_t *src, size_t bytes, bool to_host, hipStream_t st, bool beside, hipError_t *err)
    {
        std::unique_lock<std::mutex> own(busy, std::try_to_lock);
        if (!own.owns_lock()) return false;
        hipError_t e = beside ? hipSuccess : hipEventRecord(start, st);
        if (e == hipSuccess) {
            std::unique_lock<std::mutex> lk(mu);
            job = Job{dst, src, bytes, to_host, beside};
            next = 0;
            error = hipSuccess;
            left = (int)threads.size();
            ++generation;
            lk.unlock();
            cv_job.notify_all();
            work(lanes.back());  // the caller takes part
            lk.lock();
            cv_done.wait(lk, [&] { return left == 0; });
            e = error;
        }
        *err = e;
        return true;
    }

private:
    struct Job {
        uint8_t *dst;
        const uint8_t *src;
        size_t bytes;
        bool to_host, beside;
    };
    bool ok = false;
    int device;
    std::vector<Lane> lanes;
    std::vector<std::thread> threads;
    std::mutex busy;  // one copy at a time
    std::mutex mu;
    std::condition_variable cv_job, cv_done;
    uint64_t generation = 0;
    int left = 0;
    bool quit = false;
    Job job{};
    std::atomic<size_t> next{0};
    hipError_t error = hipSuccess;
    hipEvent_t start = nullptr;

    explicit Copier(int dev) : device(dev)
    {
        cpu_set_t set;
        int cpus = 1;
        if (sched_getaffinity(0, sizeof set, &set) == 0) cpus = CPU_COUNT(&set);
        const int n = std::max(1, std::min(kMaxCopyThreads, cpus / 2));
        bool good = hipEventCreateWithFlags(&start, hipEventDisableTiming) == hipSuccess;
        try {
            lanes.reserve(n);
            for (int i = 0; i < n && good; ++i) {
                Lane l;
                good = hipStreamCreateWithFlags(&l.st, hipStreamNonBlocking) == hipSuccess;
                for (int j = 0; j < 2 && good; ++j)
                    good = hipHostMalloc((void **)&l.slot[j], kChunk, hipHostMallocDefault) == hipSuccess &&
                           hipEventCreateWithFlags(&l.ev[j], hipEventDisableTiming) == hipSuccess;
                lanes.push_back(l);
            }
            for (int i = 0; i + 1 < n && good; ++i) threads.emplace_back([this, i] { loop(i); });
        } catch (...) {
            good = false;
        }
        ok = good;
        if (!good) (void)hipGetLastError();
    }
    ~Copier()
    {
        {
            std::lock_guard<std::mutex> lk(mu);
            quit = true;
        }
        cv_job.notify_all();
        for (auto &t : threads) t.join();
        for (Lane &l : lanes) {
            for (int j = 0; j < 2; ++j) {
                if (l.ev[j]) (void)hipEventDestroy(l.ev[j]);
                if (l.slot[j]) (void)hipHostFree(l.slot[j]);
            }
            if (l.st) (void)hipStreamDestroy(l.st);
        }
        if (start) (void)hipEventDestroy(start);
    }

    void loop(int i)
    {
        (void)hipSetDevice(device);
        uint64_t seen = 0;
        for (;;) {
            {
                std::unique_lock<std::mutex> lk(mu);
                cv_job.wait(lk, [&] { return quit || generation != seen; });
                if (quit) return;
                seen = generation;
            }
            work(lanes[i]);
            std::lock_guard<std::mutex> lk(mu);
            if (--left == 0) cv_done.notify_all();
        }
    }

    void fail(hipError_t e)
    {
        std::lock_guard<std::mutex> lk(mu);
        if (error == hipSuccess) error = e;
    }

    // Takes chunks until none are left; returns with its stream idle.
    void work(Lane &l)
    {
        const Job j = job;
        hipError_t e = j.beside ? hipSuccess : hipStreamWaitEvent(l.st, start, 0);
        bool used[2] = {false, false};
        size_t at[2] = {0, 0}, len[2] = {0, 0};
        auto drain = [&](int s) {  // the slot's transfer is over, and for a download its bytes with the caller
            if (!used[s] || e != hipSuccess) return;
            e = hipEventSynchronize(l.ev[s]);
            if (e == hipSuccess && j.to_host) memcpy(j.dst + at[s], l.slot[s], len[s]);
            used[s] = false;
        };
        for (int s = 0; e == hipSuccess; s ^= 1) {
            const size_t off = next.fetch_add(kChunk);
            if (off >= j.bytes) break;
            drain(s);
            if (e != hipSuccess) break;
            at[s] = off;
            len[s] = std::min(kChunk, j.bytes - off);
            if (!j.to_host) memcpy(l.slot[s], j.src + off, len[s]);
            e = hipMemcpyAsync(j.to_host ? (void *)l.slot[s] : (void *)(j.dst + off),
                               j.to_host ? (const void *)(j.src + off) : (const void *)l.slot[s], len[s],
                               j.to_host ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice, l.st);
            if (e == hipSuccess) e = hipEventRecord(l.ev[s], l.st);
            used[s] = true;
            if (e == hipSuccess && j.to_host) drain(s ^ 1);
        }
        drain(0);
        drain(1);
        if (e != hipSuccess) {
            (void)hipStreamSynchronize(l.st);
            fail(e);
        }
    }
};

// Whether p is memory the runtime does not know: ordinary host memory, which
// the CPU may touch and the DMA engine may not.
bool pageable(const void *p)
{
    hipPointerAttribute_t a;
    memset(&a, 0, sizeof a);
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

int copy(void *dst, const void *src, size_t bytes, bool to_host, hipStream_t st, bool beside)
{
    if (bytes >= (to_host || beside ? kStageDown : kStageUp) && pageable(to_host ? dst : src)) {
        int dev = 0;
        HIP_OK(hipGetDevice(&dev));
        Copier *c = nullptr;
        try {
            c = Copier::get(dev);
        } catch (...) {  // no host memory for it: the runtime's copy
        }
        hipError_t e = hipSuccess;
        if (c && c->run((uint8_t *)dst, (const uint8_t *)src, bytes, to_host, st, beside, &e)) {
            if (e == hipSuccess) return 0;
            ipfe_set_error("copy of %zu bytes failed: %s", bytes, hipGetErrorString(e));
            return -1;
        }
    }
    HIP_OK(hipMemcpyAsync(dst, src, bytes, to_host ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice, st));
    return 0;
}

}  // namespace

int copy_to_host(void *dst, const void *src, size_t bytes, hipStream_t st)
{
    return copy(dst, src, bytes, true, st, false);
}
int copy_to_device(void *dst, const void *src, size_t bytes, hipStream_t st)
{
    return copy(dst, src, bytes, false, st, false);
}
int copy_to_device_beside(void *dst, const void *src, size_t bytes, hipStream_t st)
{
    return copy(dst, src, bytes, false, st, true);
}

}  // namespace ipfe
