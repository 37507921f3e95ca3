// The library's device blocks and staged copies (cufe_amd/csrc/xfer.cpp) over a
// HIP runtime of this file's own, on the CPU: what the pool asks the driver for,
// hands out, waits for and frees.  One check a run, named by argv[1]; the first
// failed expectation ends the program with status 1.
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

// device functions that the included headers mention
static inline uint32_t __umulhi(uint32_t a, uint32_t b) { return (uint32_t)(((uint64_t)a * b) >> 32); }
static inline uint64_t __umul64hi(uint64_t a, uint64_t b) { return (uint64_t)(((unsigned __int128)a * b) >> 64); }

#include "../../cufe_amd/csrc/xfer.cpp"

namespace {
struct Driver {
    std::mutex mu;
    size_t card = (size_t)288 << 30, used = 0, largest = 0;
    bool backed = false;  // blocks are real memory (for copies)
    std::map<void *, std::pair<size_t, int>> blocks;
    std::vector<void *> freed;  // in order
    uintptr_t next = 0x7000000000ull;
    int device = 0, mallocs = 0, syncs[4] = {};
    std::atomic<int> copies{0};
} drv;
std::string last_error;

#define EXPECT(c)                                                      \
    do {                                                               \
        if (!(c)) {                                                    \
            fprintf(stderr, "%s:%d: %s\n", __FILE__, __LINE__, #c);    \
            exit(1);                                                   \
        }                                                              \
    } while (0)

// this thread's allocations still to succeed; -1: all of them
thread_local long allow = -1;
struct Fed {  // this file's own records, whatever the library may allocate
    long left = allow;
    Fed() { allow = -1; }
    ~Fed() { allow = left; }
};
}  // namespace

void *operator new(size_t n)
{
    if (allow == 0) throw std::bad_alloc();
    if (allow > 0) --allow;
    void *p = malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

void ipfe_set_error(const char *fmt, ...)
{
    Fed fed;
    char b[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(b, sizeof b, fmt, ap);
    va_end(ap);
    last_error = b;
}

extern "C" {
hipError_t hipGetDevice(int *d) { *d = drv.device; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipDeviceSynchronize(void) { ++drv.syncs[drv.device]; return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n)
{
    Fed fed;
    std::lock_guard<std::mutex> lk(drv.mu);
    if (drv.used + n > drv.card) return hipErrorOutOfMemory;
    ++drv.mallocs;
    drv.used += n;
    *p = drv.backed ? malloc(n) : (void *)drv.next;
    drv.next += n + 4096;
    drv.blocks[*p] = {n, drv.device};
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    Fed fed;
    std::lock_guard<std::mutex> lk(drv.mu);
    EXPECT(drv.blocks.count(p));
    drv.used -= drv.blocks[p].first;
    if (drv.backed) free(p);
    drv.blocks.erase(p);
    drv.freed.push_back(p);
    return hipSuccess;
}
// streams run their work at once
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free((void *)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free((void *)s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = malloc(n); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) { a->type = hipMemoryTypeUnregistered; return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); ++drv.copies; return hipSuccess; }
}

namespace {
using namespace ipfe;
constexpr size_t KiB = 1 << 10, MiB = 1 << 20, GiB = (size_t)1 << 30;

void *take(size_t bytes, bool exact = false)
{
    void *p = nullptr;
    EXPECT(dev_alloc(&p, bytes, exact) == 0 && p);
    EXPECT(drv.blocks.count(p) && drv.blocks[p].first >= bytes);
    return p;
}
size_t size_of(void *p) { return drv.blocks[p].first; }

// what a new block costs, and which kept block a request takes
void sizes()
{
    const size_t some[] = {1, 511, 512, 513, 4095, 4097, 100 * KiB + 1, MiB + 1, 5 * MiB - 1, 33 * MiB + 1, 64 * MiB,
                           64 * MiB + 1, 100 * MiB + 3, GiB + 1, 4 * GiB + 1, 257 * GiB + 1};
    for (size_t n : some) {
        void *p = take(n);
        EXPECT(size_of(p) <= n + n / 8 + 511);
        EXPECT(n <= 64 * MiB || size_of(p) < n + 512);
        dev_free(p);
        dev_trim();
        p = take(n, true);
        EXPECT(size_of(p) < n + 512);
        dev_free(p);
        dev_trim();
        EXPECT(drv.used == 0);
    }
    void *a = take(900 * KiB);
    dev_free(a);
    void *b = take(899 * KiB);  // calls of about one size share a block
    EXPECT(a == b);
    dev_free(b);
    b = take(800 * KiB, true);  // not an exact request
    EXPECT(a != b && size_of(b) == 800 * KiB);
    dev_free(b);
    void *c = take(200 * MiB);
    dev_free(c);
    void *d = take(180 * MiB);
    EXPECT(c == d);
    dev_free(d);
    d = take(150 * MiB);  // a kept block more than an eighth larger stays
    EXPECT(c != d);
    void *e = take(180 * MiB, true);
    EXPECT(c != e && size_of(e) == 180 * MiB);
    void *f = take(200 * MiB, true);
    EXPECT(c == f);
}

// a row store of arrays that fit the card by their own sizes; and a request
// that only fits when everything kept is given back and nothing is rounded
void card()
{
    std::vector<void *> v;
    for (size_t n : {87 * GiB + 1, 87 * GiB + 1, 74 * GiB, 16 * GiB, 2 * GiB}) v.push_back(take(n, true));
    for (void *p : v) dev_free(p);
    dev_trim();
    EXPECT(drv.used == 0);
    void *p = take(257 * GiB);
    dev_free(p);
    drv.card = 70 * MiB;
    p = take(30 * MiB);
    void *q = take(30 * MiB);
    dev_free(p);
    p = take(40 * MiB - 512);
    EXPECT(drv.used <= drv.card);
    void *r = nullptr;
    EXPECT(dev_alloc(&r, MiB, false) != 0 && !r);
    EXPECT(last_error.find("hipMalloc of 1048576 bytes") == 0);
    dev_free(q);
    dev_free(p);
}

// a block is waited for on its own device before it is handed out again
void devices()
{
    void *a[2];
    for (drv.device = 0; drv.device < 2; ++drv.device) a[drv.device] = take(MiB);
    for (int d : {0, 1}) dev_free(a[d]);
    for (drv.device = 0; drv.device < 2; ++drv.device) {
        EXPECT(drv.syncs[drv.device] == 0);
        EXPECT(take(MiB) == a[drv.device]);
        EXPECT(drv.syncs[drv.device] == 1);
    }
    drv.device = 1;
    dev_free(a[0]);  // device 0's, released with device 1 current
    EXPECT(take(MiB) != a[0]);
    drv.device = 0;
    EXPECT(take(MiB) == a[0] && drv.syncs[0] == 2);
    // one wait covers every block released before it
    void *p[3] = {take(2 * MiB), take(3 * MiB), take(5 * MiB)};
    for (void *q : p) dev_free(q);
    EXPECT(take(5 * MiB) == p[2] && take(2 * MiB) == p[0] && take(3 * MiB) == p[1] && drv.syncs[0] == 3);
}

// beyond 4 GiB kept, the blocks released longest ago are freed, and calls of a
// size not seen before find their blocks again
void bound()
{
    std::vector<void *> v;
    for (int i = 0; i < 9; ++i) v.push_back(take(512 * MiB + 512 * i));
    for (void *p : v) dev_free(p);
    EXPECT(drv.freed == std::vector<void *>({v[0], v[1]}));  // seven of them stay below 4 GiB
    EXPECT(drv.used <= 4 * GiB);
    const int mallocs = drv.mallocs;
    for (int i = 0; i < 5; ++i) {
        void *p = take(100 * MiB);
        dev_free(p);
    }
    EXPECT(drv.mallocs == mallocs + 1 && drv.used <= 4 * GiB);
    void *p = take(450 * MiB);
    dev_free(p);
    EXPECT(drv.freed == std::vector<void *>({v[0], v[1], v[2]}) && take(450 * MiB) == p);
    dev_free(p);
    p = take(4 * GiB + 1);  // never kept, and nothing goes for it
    dev_free(p);
    EXPECT(drv.freed.size() == 4 && drv.freed.back() == p);
    p = take(4 * GiB);
    dev_free(p);
    EXPECT(drv.used == 4 * GiB && take(4 * GiB) == p);
    dev_free(p);
    dev_trim();
    EXPECT(drv.used == 0 && drv.blocks.empty());
    dev_free(nullptr);
}

// f with n allocations left
template <class F>
auto starved(long n, F f)
{
    allow = n;
    auto r = f();
    allow = -1;
    return r;
}

// host memory that runs out is an error, and no block is lost or ends the process
void starve()
{
    for (int n = 0; n < 4; ++n) {
        void *p = (void *)1;
        if (starved(n, [&] { return dev_alloc(&p, MiB); })) {
            EXPECT(!p && drv.used == 0);
            EXPECT(last_error.find("no host memory") == 0);
        } else {
            EXPECT(p && size_of(p) == MiB);
            starved(0, [&] { dev_free(p); return 0; });  // cannot be recorded: freed
            EXPECT(drv.used == 0);
        }
    }
    void *p = take(MiB);
    dev_free(p);
    EXPECT(take(MiB) == p);  // the records are sound
    // a copy that cannot have its threads goes through the runtime
    drv.backed = true;
    std::vector<uint8_t> a(9 * MiB, 7), b(9 * MiB);
    EXPECT(starved(0, [&] { return copy_to_device(b.data(), a.data(), a.size(), nullptr); }) == 0);
    EXPECT(a == b);
}

// where a copy goes through the threads' chunks (2 MiB each) and where in one
void paths()
{
    std::vector<uint8_t> a(8 * MiB, 3), b(8 * MiB);
    auto transfers = [&](auto copy, size_t n) {
        const int before = drv.copies;
        EXPECT(copy(b.data(), a.data(), n, nullptr) == 0);
        return drv.copies - before;
    };
    EXPECT(transfers(copy_to_host, 4 * MiB - 1) == 1 && transfers(copy_to_host, 4 * MiB) == 2);
    EXPECT(transfers(copy_to_device, 8 * MiB - 1) == 1 && transfers(copy_to_device, 8 * MiB) == 4);
    EXPECT(transfers(copy_to_device_beside, 4 * MiB - 1) == 1 && transfers(copy_to_device_beside, 4 * MiB) == 2);
}

// large copies of several threads at once, each to and from its own arrays: all
// end, with their own bytes, whichever of them has the copy threads
void copies()
{
    std::atomic<int> done{0};
    std::vector<std::thread> t;
    for (int k = 0; k < 6; ++k)
        t.emplace_back([k, &done] {
            for (int i = 0; i < 12; ++i) {
                const size_t n = 8 * MiB + (size_t)k * 777777 + i * 131071;
                std::vector<uint8_t> a(n), b(n), c(n);
                for (size_t j = 0; j < n; ++j) a[j] = (uint8_t)(j * 31 + j / 4096 + k + i);
                EXPECT((i & 1 ? copy_to_device : copy_to_device_beside)(b.data(), a.data(), n, nullptr) == 0);
                EXPECT(copy_to_host(c.data(), b.data(), n, nullptr) == 0);
                EXPECT(a == b && a == c);
                ++done;
            }
        });
    for (auto &x : t) x.join();
    EXPECT(done == 72);
}
}  // namespace

int main(int argc, char **argv)
{
    const std::map<std::string, void (*)()> checks = {{"sizes", sizes}, {"card", card}, {"devices", devices}, {"bound", bound},
                                                      {"starve", starve}, {"copies", copies}, {"paths", paths}};
    EXPECT(argc == 2 && checks.count(argv[1]));
    checks.at(argv[1])();
    printf("%s ok\n", argv[1]);
    fflush(stdout);
    _Exit(0);
}
