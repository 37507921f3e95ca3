// k_gauss_walk.hip -- call boundaries of the Gaussian streams from the
// per-chunk accept counts (the second pass of k_sampler.hip).
//
// A call starts on the chunk after the previous call's last one and ends on
// the first chunk that brings its accepted candidates to slen, so call k's
// start depends on every call before it.  Only where a stream enters a window
// of chunks depends on what came before, and it enters within one call's span
// of the window's start.  Three launches therefore cut the chain:
//   1. map:   every window of WALK_WIN chunks, in parallel: for each chunk the
//             stream could enter it at, the calls that start in the window and
//             where the next one starts after it;
//   2. chain: one thread per stream follows the maps from window to window;
//   3. fill:  every window, in parallel: its calls from its true entry, and
//             the labels of its chunks.
// One wave per stream walking all its calls in order (5.2 us a call, whatever
// the number of streams) took 4.07 ms for the 785 calls of one message at the
// reference's key length, seven times the candidates before it; the three
// launches take 0.07 ms (the whole call went from 11.1 to 7.2 ms).  Where every
// stream fits one window its entry is chunk 0 and the third launch does alone
// (one call of S1: 4.5 us, 21.5 in three launches).
#include "kernels.h"

namespace ipfe {

namespace {

constexpr int WALK_WIN = GAUSS_WALK_WIN;
constexpr int WALK_THREADS = 512;
constexpr int WALK_SLAB = 8 * WALK_THREADS;  // chunks scanned at a time
// the most chunks a call may span (GaussStream::span, at most slen / 2)
constexpr int WALK_HALO = 4096;
constexpr int WALK_RUN = WALK_WIN / WALK_THREADS + 1;  // consecutive chunks of a thread of the map pass
constexpr int WALK_STARTS = WALK_WIN / 256 + 1;  // calls starting in a window: 256 chunks at least for slen 2048
static_assert((WALK_WIN + WALK_HALO) % WALK_SLAB == 0, "whole slabs");

// Inclusive prefix sums, mod 2^16, of `need` counts into P (differences over
// at most WALK_HALO chunks are below 2^15).  Counts from `avail` on are 0.
// The counts are read 8 at a time; the plan pads every stream to 16 chunks.
__device__ void walk_scan(const uint8_t *__restrict__ cnt, int avail, int need, uint16_t *P, uint32_t (*wsum)[8])
{
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    uint32_t carry = 0;
    for (int s = 0, b = 0; s < need; s += WALK_SLAB, b ^= 1) {
        const int i0 = s + 8 * tid;
        uint2 v = make_uint2(0, 0);
        if (i0 < avail && i0 < need) v = *reinterpret_cast<const uint2 *>(cnt + i0);
        uint32_t l[8], sum = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t c = ((j < 4 ? v.x : v.y) >> (8 * (j & 3))) & 255u;
            sum += i0 + j < avail ? c : 0u;
            l[j] = sum;
        }
        uint32_t incl = sum;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(incl, d, 64);
            if (lane >= d) incl += o;
        }
        if (lane == 63) wsum[b][wv] = incl;
        __syncthreads();
        uint32_t before = carry + incl - sum;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t t = wsum[b][j];
            before += j < wv ? t : 0u;
            carry += t;
        }
        if (i0 < need) {
            uint32_t w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = ((before + l[2 * j]) & 0xffffu) | ((before + l[2 * j + 1]) << 16);
            *reinterpret_cast<uint4 *>(P + i0) = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
    __syncthreads();
}

// accepted candidates of chunks [c, i] and those before c
__device__ __forceinline__ uint32_t walk_ex(const uint16_t *P, int c) { return c ? P[c - 1] : 0u; }
__device__ __forceinline__ uint32_t walk_sum(const uint16_t *P, uint32_t ex, int i) { return (P[i] - ex) & 0xffffu; }

struct WalkWindow {
    int w, nwin, avail, need, span;
    uint32_t *slot;  // the window's map, later its entry
    __device__ WalkWindow(const GaussStream *S, int w_, int *pos, uint32_t *map) : w(w_)
    {
        span = S->span;
        avail = S->nchunks - w * WALK_WIN;
        nwin = min(WALK_WIN, avail);
        need = min(avail, WALK_WIN + span);
        // full streams: the labels the fill pass writes later have room for
        // the map; compact streams have no labels and a map of their own
        slot = S->coef0_only ? map + S->map_base + (long long)w * span
                             : reinterpret_cast<uint32_t *>(pos + S->chunk_base + (long long)w * WALK_WIN);
    }
};

// Map word of an entry chunk: bits 0..12 the next window's entry, 13..15 the
// last call's candidates beyond slen (0..7), 16..23 calls that start in the
// window and end, bit 31 when the last of them does not end in the chunks read.
constexpr uint32_t WALK_OPEN = 0x80000000u;

__global__ __launch_bounds__(WALK_THREADS) void k_walk_map(const GaussStream *__restrict__ streams, int maxw,
                                                            const uint8_t *__restrict__ cnt, int *__restrict__ pos,
                                                            uint32_t *__restrict__ map)
{
    __shared__ __align__(16) uint16_t P[WALK_WIN + WALK_HALO];
    __shared__ uint16_t next[WALK_WIN];
    __shared__ uint32_t wsum[2][8];
    const GaussStream *S = streams + blockIdx.x / maxw;
    const int w = (int)(blockIdx.x % maxw);
    if ((long long)w * WALK_WIN >= S->nchunks) return;
    const WalkWindow W(S, w, pos, map);
    const uint32_t slen = (uint32_t)S->slen;
    walk_scan(cnt + S->chunk_base + (long long)w * WALK_WIN, W.avail, W.need, P, wsum);
    // Where the call that starts at each chunk ends: a thread takes WALK_RUN
    // consecutive chunks, whose ends follow one another, and searches only for
    // the first (25 us for a message of 785 slots; a search per entry and
    // call took 49).  An odd run keeps the
    // lanes' addresses off each other's banks.
    {
        int lo = 0;
        for (int c = WALK_RUN * threadIdx.x, u = 0; u < WALK_RUN && c < W.nwin; ++u, ++c) {
            const uint32_t ex = walk_ex(P, c);
            int hi = min(c + W.span, W.need) - 1;
            lo = max(lo, c + (int)slen / 8 - 1);
            uint32_t n = 0;
            if (lo <= hi && walk_sum(P, ex, hi) >= slen) {
                if (u == 0)
                    while (lo < hi) {
                        const int mid = (lo + hi) >> 1;
                        if (walk_sum(P, ex, mid) >= slen) hi = mid; else lo = mid + 1;
                    }
                else
                    while (walk_sum(P, ex, lo) < slen) ++lo;
                n = (uint32_t)(lo + 1 - c);
            }
            next[c] = (uint16_t)n;
        }
    }
    __syncthreads();
    const int entries = w == 0 ? 1 : min(W.span, W.nwin);
    for (int o = threadIdx.x; o < entries; o += WALK_THREADS) {
        int c = o, last = o;
        uint32_t calls = 0, open = 0;
        while (c < W.nwin) {
            const uint32_t n = next[c];
            if (n == 0) {
                open = WALK_OPEN;
                break;
            }
            last = c;
            c += (int)n;
            ++calls;
        }
        const uint32_t over = calls ? walk_sum(P, walk_ex(P, last), c - 1) - slen : 0u;
        W.slot[o] = open | (uint32_t)max(0, c - WALK_WIN) | over << 13 | calls << 16;
    }
}

// One thread per stream.  Leaves in slot 0 of each window bits 0..12 its
// entry, 13..15 the excess of the call that ends there, bit 31 when no call of
// the stream has chunks in it, and in slot 1 the call that starts at the entry.
__global__ void k_walk_chain(const GaussStream *__restrict__ streams, int nstreams, int *__restrict__ pos,
                             uint32_t *__restrict__ map, int *__restrict__ status)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nstreams) return;
    const GaussStream *S = streams + s;
    const int ncalls = S->ncalls, nw = (S->nchunks + WALK_WIN - 1) / WALK_WIN;
    int o = 0, k = 0;
    uint32_t over = 0;
    bool open = false;
    for (int w = 0; w < nw; ++w) {
        const WalkWindow W(S, w, pos, map);
        const bool used = !open && (k < ncalls || (k == ncalls && o > 0));
        uint32_t word = WALK_OPEN;
        if (used && k < ncalls && o < W.nwin) word = W.slot[o];
        W.slot[0] = used ? (uint32_t)o | over << 13 : WALK_OPEN;
        W.slot[1] = (uint32_t)k;
        open = open || (word & WALK_OPEN) != 0;
        k += (int)((word >> 16) & 255u);
        o = (int)(word & 0x1fffu);
        over = (word >> 13) & 7u;
    }
    if (k < ncalls) status[s] = 1;
}

// Full streams: pos[chunk] = call << 13 | first output position, or -1.
// Compact streams: firsts of the calls that start in the window.  one: the
// streams have one window each and no map was made.
__global__ __launch_bounds__(WALK_THREADS) void k_walk_fill(const GaussStream *__restrict__ streams, int maxw,
                                                             const uint8_t *__restrict__ cnt, int *__restrict__ pos,
                                                             uint32_t *__restrict__ map,
                                                             long long *__restrict__ firsts, int one,
                                                             int *__restrict__ status)
{
    __shared__ __align__(16) uint16_t P[WALK_WIN + WALK_HALO];
    __shared__ uint32_t wsum[2][8];
    __shared__ int start[WALK_STARTS + 1];
    __shared__ int s_n;
    const GaussStream *S = streams + blockIdx.x / maxw;
    const int w = (int)(blockIdx.x % maxw), tid = threadIdx.x, lane = tid & 63;
    if ((long long)w * WALK_WIN >= S->nchunks) return;
    const WalkWindow W(S, w, pos, map);
    const bool compact = S->coef0_only != 0;
    const long long base = S->chunk_base + (long long)w * WALK_WIN;
    const uint32_t entry = one ? 0u : W.slot[0], slen = (uint32_t)S->slen;
    const int k = one ? 0 : (int)W.slot[1];
    const int npad = (W.nwin + 15) & ~15;  // the plan's padding carries no call
    if (entry & WALK_OPEN) {
        __syncthreads();  // every thread has read the slots
        if (!compact)
            for (int i = tid; i < npad; i += WALK_THREADS) pos[base + i] = -1;
        return;
    }
    const int o = (int)(entry & 0x1fffu), ncalls = S->ncalls;
    walk_scan(cnt + base, W.avail, W.need, P, wsum);
    if (tid < 64) {
        // the first wave finds each call's end in two 64-way steps
        int c = o, n = 0;
        while (c < W.nwin && k + n < ncalls && n < WALK_STARTS) {
            const uint32_t ex = walk_ex(P, c);
            const int lo = c + (int)slen / 8 - 1, hi = min(c + W.span, W.need) - 1;
            if (lo > hi) break;
            const int st = (hi - lo) / 64 + 1, p = min(lo + st * (lane + 1) - 1, hi);
            const uint64_t a = __ballot(walk_sum(P, ex, p) >= slen);
            if (!a) break;
            const int q0 = lo + st * (__ffsll((unsigned long long)a) - 1), q = min(q0 + lane, hi);
            const uint64_t b = __ballot(walk_sum(P, ex, q) >= slen);
            if (lane == 0) start[n] = c;
            ++n;
            c = q0 + __ffsll((unsigned long long)b);  // one past the call's last chunk
        }
        if (lane == 0) {
            start[n] = c;
            s_n = n;
            if (one && n < ncalls) status[blockIdx.x] = 1;
        }
    }
    __syncthreads();
    const int n = s_n, end = start[n];
    if (compact) {
        if (tid < n) {
            int i = start[tid];
            const uint32_t ex = walk_ex(P, i);
            while (walk_sum(P, ex, i) == 0) ++i;  // ends: the call has slen accepted candidates
            firsts[S->first_base + k + tid] = base + i;
        }
        return;
    }
    const uint32_t total = slen + ((entry >> 13) & 7u), oex = o ? P[o - 1] : 0u;
    for (int i0 = 4 * tid; i0 < npad; i0 += 4 * WALK_THREADS) {
        int lo = 0, hi = n;  // the first call that starts after i0
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (start[mid] > i0) hi = mid; else lo = mid + 1;
        }
        int4 out;
        int *po = &out.x;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = i0 + u;
            if (lo < n && start[lo] <= i) ++lo;
            int label = -1;
            if (i < o)
                label = (int)((uint32_t)(k - 1) << 13 | ((total - ((oex - walk_ex(P, i)) & 0xffffu)) & 0x1fffu));
            else if (i < end && lo > 0)
                label = (int)((uint32_t)(k + lo - 1) << 13 | ((walk_ex(P, i) - walk_ex(P, start[lo - 1])) & 0xffffu));
            po[u] = label;
        }
        *reinterpret_cast<int4 *>(pos + base + i0) = out;
    }
}

}  // namespace

int launch_gauss_walk(const GaussStream *d_streams, int nstreams, int max_chunks, const uint8_t *cnt, int *pos,
                      uint32_t *map, long long *firsts, int *status, hipStream_t st)
{
    if (nstreams <= 0) return 0;
    const int maxw = (max_chunks + WALK_WIN - 1) / WALK_WIN;
    const long long blocks = (long long)nstreams * maxw;
    // a launch takes fewer than 2^32 threads (a group of 2^28 chunks at most, with
    // streams of up to 65 windows beside the shortest: half of that)
    if (maxw < 1 || blocks >= (1ll << 32) / WALK_THREADS) {
        ipfe_set_error("Gaussian walk: %d streams of up to %d chunks", nstreams, max_chunks);
        return -1;
    }
    if (maxw > 1) {
        hipLaunchKernelGGL(k_walk_map, dim3((unsigned)blocks), dim3(WALK_THREADS), 0, st, d_streams, maxw, cnt, pos,
                           map);
        hipLaunchKernelGGL(k_walk_chain, dim3((unsigned)((nstreams + 63) / 64)), dim3(64), 0, st, d_streams, nstreams,
                           pos, map, status);
    }
    hipLaunchKernelGGL(k_walk_fill, dim3((unsigned)blocks), dim3(WALK_THREADS), 0, st, d_streams, maxw, cnt, pos, map,
                       firsts, maxw == 1, status);
    HIP_OK(hipGetLastError());
    return 0;
}

}  // namespace ipfe
