// runtime.h -- device state shared by the C ABI: uploaded constant tables,
// device buffers with RAII, and the Gaussian-sampler driver.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <functional>
#include <utility>
#include <vector>

#include "host_tables.h"
#include "kernels.h"

namespace ipfe {

extern const uint32_t *g_aes_te;

// Per-process device state (one GPU, the one current at the library's first
// call): constant tables resident in HBM, in static device arrays (set-up
// allocates nothing).
struct Device {
    int id = 0;                  // the HIP device the state belongs to
    uint32_t *tw_all = nullptr;  // [4][3][N]
    uint32_t *aes_te = nullptr;  // [1024]
    NinvConsts ninv;
    ScaleConsts scale;
    BarrettConsts barrett;
    hipStream_t stream = nullptr;
};
// Initialises on first use; returns nullptr (error set) on failure.
Device *device();

// A device block of at least `bytes` bytes, uninitialised, and its release.
// Released blocks are kept for the next allocation (xfer.cpp): bounded, from
// any thread; a block is not handed out again before the device has finished
// the work issued before its release.  exact: a block of that size (to 512 bytes),
// for buffers that stay; others may be an eighth larger.
int dev_alloc(void **out, size_t bytes, bool exact = false);
void dev_free(void *p);
// Frees the blocks kept.
void dev_trim();

// Copies between device memory and the caller's, after the work st holds; what
// st is given later follows a copy_to_device.  Large copies to or from
// pageable memory are done when they return; the others when st is (as
// hipMemcpyAsync).  Not for a stream that is being captured.
int copy_to_host(void *dst, const void *src, size_t bytes, hipStream_t st);
int copy_to_device(void *dst, const void *src, size_t bytes, hipStream_t st);
// copy_to_device into a block no work has been given yet: a large pageable copy
// runs beside what st holds, instead of after it.
int copy_to_device_beside(void *dst, const void *src, size_t bytes, hipStream_t st);

template <typename T>
struct DevBuf {
    T *p = nullptr;
    size_t n = 0;
    DevBuf() = default;
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    DevBuf &operator=(DevBuf &&o)
    {
        reset();
        swap(o);
        return *this;
    }
    ~DevBuf() { reset(); }
    void reset()
    {
        dev_free(p);
        p = nullptr;
        n = 0;
    }
    int alloc(size_t count, bool exact = false)
    {
        reset();
        if (count == 0) return 0;
        if (dev_alloc((void **)&p, count * sizeof(T), exact)) return -1;
        n = count;
        return 0;
    }
    T *get() const { return p; }
    void swap(DevBuf &o)
    {
        std::swap(p, o.p);
        std::swap(n, o.n);
    }
};

// One Gaussian stream request for the sampler driver.
struct StreamReq {
    uint32_t rk[60];
    uint16_t nonce;
    int which;  // sampler width index (GaussStream::which)
    int ncalls;
    uint32_t *out0;
    uint32_t *out1;
    long long out_stride;
    int coef0_only;
    int slen;          // samples per call
    int nmod;          // output limbs and their moduli / fold shifts
    uint32_t q[4], fold[4];
};
// A stream of the reference parameter set (4096 samples per call, 3 limbs);
// which = 1, 2, 3 for S1, S2, S3.
StreamReq make_stream(const uint8_t key[32], uint16_t nonce, int which, int ncalls, uint32_t *out0, uint32_t *out1,
                      long long out_stride, int coef0_only = 0);
struct PsetSpec;
// A stream of parameter set ps: sampler which = 1, 2, 3 at that set's widths.
StreamReq make_stream_ps(const PsetSpec &ps, const uint8_t key[32], uint16_t nonce, int which, int ncalls,
                         uint32_t *out0, uint32_t *out1, long long out_stride);

constexpr size_t kGaussScratch = (size_t)8 << 30;
// Samples every request (device outputs), bit-exact with the reference
// sequential sampler; splits into groups that fit scratch_budget bytes.  beside
// (if given) is called once, with the first group's kernels launched and their
// outcome not yet awaited, for host work that should overlap them.
int run_gauss(const std::vector<StreamReq> &reqs, hipStream_t st, size_t scratch_budget = kGaussScratch,
              const std::function<int()> &beside = {});

// One group of sampler streams, split into host planning, table upload, the
// kernel launches (no host round trip, so a graph can capture them) and the
// status check that reports a speculative window that was too short.
struct GaussPlan {
    int n = 0, level = 0;
    int full = 0;  // scan a chunk past its default AES blocks (set after one needed it)
    long long chunks = 0, full_chunks = 0, nfirst = 0;
    long long map_words = 0;  // of the walk's maps of the compact streams
    int max_chunks = 0;
    std::vector<GaussStream> hs;
    std::vector<long long> chunk_prefix, first_prefix;
    DevBuf<GaussStream> d_streams;
    DevBuf<long long> d_cp, d_fp, d_first;
    DevBuf<int> d_status;
    // device metadata the kernels read: the buffers above, or a region bound
    // with bind_meta
    GaussStream *m_streams = nullptr;
    long long *m_cp = nullptr, *m_fp = nullptr, *m_first = nullptr;
    int *m_status = nullptr;
    DevBuf<uint8_t> own_cnt;
    DevBuf<uint64_t> own_vals;
    DevBuf<int> own_pos;
    uint8_t *s_cnt = nullptr;
    uint64_t *s_vals = nullptr;
    int *s_pos = nullptr;
    uint32_t *s_map = nullptr;  // the walk's maps of the compact streams

    // alloc_meta false: plan only; the caller binds the device metadata
    // (bind_meta) and the chunk scratch (bind_scratch_region) to its memory
    // (plans of full streams only: the walk's maps of compact streams come
    // with alloc_scratch)
    int build(const StreamReq *reqs, int n, int level, bool alloc_meta = true);
    size_t meta_bytes() const;
    int bind_meta(uint8_t *base);
    // the chunk scratch as one region of 256-byte aligned pieces
    size_t bound_scratch_bytes() const;
    int bind_scratch_region(uint8_t *base);
    // chunk scratch: own allocation, or a caller's buffers (a count per chunk;
    // 8 values and a position per full-stream chunk)
    int alloc_scratch();
    int bind_scratch(uint8_t *cnt, uint64_t *vals, int *pos);
    void rekey(const StreamReq *reqs);
    int upload(hipStream_t st);
    int launch(hipStream_t st);
    // overflow: a window was short; need_full: a chunk needed AES blocks the
    // default set leaves out (rerun with full = 1)
    int check(hipStream_t st, int *overflow, int *need_full);
};

// Speculative window (chunks) for a stream of ncalls calls of slen samples of
// sampler width `which` at margin level m, and the scratch bytes one stream
// needs at level 0 (the three-argument forms: 4096 samples per call).
long long gauss_window(int which, int slen, int ncalls, int m);
long long gauss_window(int which, int ncalls, int m);
size_t gauss_bytes(int which, int slen, int ncalls, int coef0_only);
size_t gauss_bytes(int which, int ncalls, int coef0_only);

int sync_stream(hipStream_t st);

// [p, p + bytes) lies inside one block from cufe_host_alloc (pinned).
bool host_pinned(const void *p, size_t bytes);

}  // namespace ipfe
