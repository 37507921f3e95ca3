// k_scheme.hip -- functional-key generation, the sum part of decryption and
// CRT + rounding, bit-exact with src/rlwe_sife.c:215-393 and src/crt.c:46-82.
//
// Keygen and the first half of decryption fold  acc <- mod_prime(y_i v_i + acc)
// over every slot i < L in order (src/rlwe_sife.c:232-240, :265-273).  Here it
// is computed as a plain sum: mod_prime returns the canonical residue unless
// its argument is a multiple of the modulus, so the fold's result is the
// canonical sum wherever that is not zero.  Where it is zero the result is 0 or
// q by the fold's last steps (fold_zero).  The sum takes one 64-bit multiply-add
// a term (two for y of 16 bits and more: the halves of y apart; 785 terms stay
// below 2^57) and one reduction at the end, in any order, where the fold is a
// chain of data-dependent loops -- 65 us for one vector of 123 terms.
#include <algorithm>

#include "crt_dev.h"
#include "fold_dev.h"
#include "kernels.h"

namespace ipfe {

// y_v[i] mod q_s as the fold takes it; below 2^16 it is y itself
__device__ __forceinline__ uint32_t fold_y(uint32_t y, int s) { return y >> 16 ? mod_prime_exact(y, s) : y; }

// fold_zero of vector v at the coefficient base points at
__device__ uint32_t fold_zero_sparse(const SparseY &y, int v, int s, const uint32_t *base)
{
    const int e0 = y.off[v];
    return fold_zero(y.off[v + 1] - e0, y.len, qmod(s), [s](uint64_t m) { return mod_prime_exact(m, s); }, [&](int e, uint32_t &yy, uint32_t &vv, int &i) {
        i = y.idx[e0 + e];
        yy = fold_y(y.val[e0 + e], s);
        vv = base[(size_t)i * 3 * IPFE_N];
    });
}

// Few sparse vectors: 64 coefficients a workgroup, the entries dealt to four
// waves, so that one vector's 12,288 chains are 768 waves of a quarter of the
// terms (65 us -> 10.5 for one of 123).  Grid (3 N / 64, nvec).
__global__ __launch_bounds__(64 * FOLD_WAVES) void k_fold_few(SparseY y, const uint32_t *__restrict__ P,
                                                             uint32_t *__restrict__ out, BarrettConsts bc)
{
    __shared__ uint32_t part[FOLD_WAVES][64];
    const int v = blockIdx.y, s = blockIdx.x / (IPFE_N / 64), lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int k = (int)(blockIdx.x % (IPFE_N / 64)) * 64 + lane;
    const uint32_t *base = P + (size_t)s * IPFE_N + k;
    const int e0 = y.off[v], e1 = y.off[v + 1];
    FoldSum acc;
#pragma unroll 8
    for (int e = e0 + w; e < e1; e += FOLD_WAVES)
        acc.add(fold_y(y.val[e], s), base[(size_t)y.idx[e] * 3 * IPFE_N]);
    part[w][lane] = acc.value(qmod(s), bc.mu_hi[s], bc.mu_lo[s]);
    __syncthreads();
    if (w) return;
    uint64_t t = 0;
#pragma unroll
    for (int j = 0; j < FOLD_WAVES; ++j) t += part[j][lane];
    uint32_t r = (uint32_t)(t % qmod(s));
    if (r == 0) r = fold_zero_sparse(y, v, s, base);
    out[((size_t)v * 3 + s) * IPFE_N + k] = r;
}

// Many sparse vectors: four consecutive coefficients a thread, 16-byte loads
// (2,000 vectors of 14 entries: 267 -> 76 us, bound by the 1.4 GB of key words
// that they read from the caches, at 18 TB/s).
// Grid (3 N / 1024, nvec).
__global__ __launch_bounds__(256) void k_fold_many(SparseY y, const uint32_t *__restrict__ P,
                                                   uint32_t *__restrict__ out, BarrettConsts bc)
{
    const int v = blockIdx.y, s = blockIdx.x / (IPFE_N / 1024);
    const int k = (int)(blockIdx.x % (IPFE_N / 1024)) * 1024 + 4 * threadIdx.x;
    const uint32_t *base = P + (size_t)s * IPFE_N + k;
    const int e0 = y.off[v], e1 = y.off[v + 1];
    FoldSum acc[4];
#pragma unroll 4
    for (int e = e0; e < e1; ++e) {
        const uint4 p = *reinterpret_cast<const uint4 *>(base + (size_t)y.idx[e] * 3 * IPFE_N);
        const uint32_t t = fold_y(y.val[e], s);
        acc[0].add(t, p.x);
        acc[1].add(t, p.y);
        acc[2].add(t, p.z);
        acc[3].add(t, p.w);
    }
    uint32_t r[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        r[u] = acc[u].value(qmod(s), bc.mu_hi[s], bc.mu_lo[s]);
        if (r[u] == 0) r[u] = fold_zero_sparse(y, v, s, base + u);
    }
    *reinterpret_cast<uint4 *>(out + ((size_t)v * 3 + s) * IPFE_N + k) = make_uint4(r[0], r[1], r[2], r[3]);
}

// Dense vectors with every y below 2^16: FOLD_VECS vectors share each word of
// P; their y come from scalar loads, a slot's 16 side by side (k_fold_pack; from
// 16 rows of y apart it took 87 us).  64 coefficients a workgroup, the slots
// dealt to four waves: 128 vectors of 785 slots in 62 us + 5 for the packing
// (1,131 for the literal fold).  Grid (3 N / 64, nvec / FOLD_VECS).
constexpr int FOLD_VECS = 16;

// y [nvec][len] -> [nvec / 16][len][16], zeros past nvec
__global__ void k_fold_pack(const uint32_t *__restrict__ y, int nvec, int len, uint32_t *__restrict__ packed)
{
    const int v = blockIdx.y * FOLD_VECS + (threadIdx.x & (FOLD_VECS - 1));
    const int i = blockIdx.x * (256 / FOLD_VECS) + threadIdx.x / FOLD_VECS;
    if (i < len) packed[((size_t)blockIdx.y * len + i) * FOLD_VECS + (threadIdx.x & (FOLD_VECS - 1))] =
        v < nvec ? y[(size_t)v * len + i] : 0u;
}

__global__ __launch_bounds__(64 * FOLD_WAVES) void k_fold_dense(const uint32_t *__restrict__ y,
                                                               const uint32_t *__restrict__ packed, int nvec,
                                                               int len, const uint32_t *__restrict__ P,
                                                               uint32_t *__restrict__ out, BarrettConsts bc)
{
    __shared__ uint32_t part[FOLD_WAVES][FOLD_VECS][64];
    const int v0 = blockIdx.y * FOLD_VECS, s = blockIdx.x / (IPFE_N / 64), lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int k = (int)(blockIdx.x % (IPFE_N / 64)) * 64 + lane;
    const uint32_t *base = P + (size_t)s * IPFE_N + k;
    const int i0 = len * w / FOLD_WAVES, i1 = len * (w + 1) / FOLD_WAVES;
    uint64_t acc[FOLD_VECS] = {};
    const uint32_t *yp = packed + (size_t)blockIdx.y * len * FOLD_VECS;
#pragma unroll 4
    for (int i = i0; i < i1; ++i) {
        const uint32_t p = base[(size_t)i * 3 * IPFE_N];
#pragma unroll
        for (int j = 0; j < FOLD_VECS; ++j) acc[j] += (uint64_t)yp[(size_t)i * FOLD_VECS + j] * p;
    }
#pragma unroll
    for (int j = 0; j < FOLD_VECS; ++j)
        part[w][j][lane] = reduce64(acc[j], qmod(s), bc.mu_hi[s], bc.mu_lo[s]);
    __syncthreads();
    for (int j = w; j < FOLD_VECS && v0 + j < nvec; j += FOLD_WAVES) {
        uint64_t t = 0;
#pragma unroll
        for (int u = 0; u < FOLD_WAVES; ++u) t += part[u][j][lane];
        uint32_t r = (uint32_t)(t % qmod(s));
        if (r == 0) {
            const uint32_t *yv = y + (size_t)(v0 + j) * len;
            r = fold_zero(len, len, qmod(s), [s](uint64_t m) { return mod_prime_exact(m, s); }, [&](int e, uint32_t &yy, uint32_t &vv, int &i) {
                i = e;
                yy = yv[e];
                vv = base[(size_t)e * 3 * IPFE_N];
            });
        }
        out[((size_t)(v0 + j) * 3 + s) * IPFE_N + k] = r;
    }
}

__global__ void k_crt_round(const uint32_t *__restrict__ d, int nvec, int coef, uint32_t *__restrict__ r)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nvec) return;
    const uint32_t *dv = d + (size_t)v * 3 * IPFE_N + coef;
    r[v] = crt_decode(dv[0], dv[IPFE_N], dv[2 * IPFE_N]);
}

// out[v][3][N] = sum_i y_v[i] P[i] with the reference's sequential fold.
// Dense form: at least FOLD_VECS vectors with a quarter of their entries set
// (a vector's own list then costs more than sharing each word of P with 15
// others).  Sparse form: from 32 vectors on their coefficients alone fill the
// GPU (96 waves each), below that the entries are split as well.
int launch_fold(const SparseY &y, int nvec, const uint32_t *P, uint32_t *out, const BarrettConsts &bc, hipStream_t st)
{
    if (nvec <= 0) return 0;
    if (y.dense) {
        const unsigned groups = (unsigned)(nvec + FOLD_VECS - 1) / FOLD_VECS;
        hipLaunchKernelGGL(k_fold_pack, dim3((y.len * FOLD_VECS + 255) / 256, groups), dim3(256), 0, st, y.dense, nvec,
                           y.len, y.dense_packed);
        hipLaunchKernelGGL(k_fold_dense, dim3(3 * IPFE_N / 64, groups), dim3(64 * FOLD_WAVES), 0, st, y.dense,
                           y.dense_packed, nvec, y.len, P, out, bc);
    } else if (nvec < 32)
        hipLaunchKernelGGL(k_fold_few, dim3(3 * IPFE_N / 64, nvec), dim3(64 * FOLD_WAVES), 0, st, y, P, out, bc);
    else
        hipLaunchKernelGGL(k_fold_many, dim3(3 * IPFE_N / 1024, nvec), dim3(256), 0, st, y, P, out, bc);
    HIP_OK(hipGetLastError());
    return 0;
}

size_t fold_packed_words(size_t nvec, size_t len) { return (nvec + FOLD_VECS - 1) / FOLD_VECS * FOLD_VECS * len; }

bool fold_dense(size_t nvec, size_t len, size_t nnz, uint32_t max_y)
{
    return nvec >= FOLD_VECS && nnz > 0 && max_y < 65536u && nnz * 4 >= nvec * len;
}

int launch_crt_round(const uint32_t *d, int nvec, int coef, uint32_t *r, hipStream_t st)
{
    if (nvec <= 0) return 0;
    hipLaunchKernelGGL(k_crt_round, dim3((nvec + 255) / 256), dim3(256), 0, st, d, nvec, coef, r);
    HIP_OK(hipGetLastError());
    return 0;
}

// Sparse lists of dense vectors y [n][stride], one wave per vector: counts (into
// off[v + 1]) with info[0] = the largest slot in use plus one and info[1] =
// v stride + i of the first entry at a slot i >= limit, then their prefix sums, then
// the entries.
__global__ __launch_bounds__(256) void k_sparse_count(const uint32_t *__restrict__ y, int n, int stride, int limit,
                                                      int *__restrict__ off, unsigned int *__restrict__ info)
{
    const int v = blockIdx.x * 4 + threadIdx.x / 64, lane = threadIdx.x & 63;
    if (v >= n) return;
    const uint32_t *row = y + (size_t)v * stride;
    int cnt = 0, last = -1;
    for (int i0 = 0; i0 < stride; i0 += 64) {
        const bool set = i0 + lane < stride && row[i0 + lane] != 0;
        const uint64_t m = __ballot(set);
        cnt += __popcll(m);
        if (m) last = i0 + 63 - __clzll((long long)m);
        const uint64_t over = __ballot(set && i0 + lane >= limit);
        if (over && lane == 0) atomicMin(info + 1, (unsigned int)v * stride + i0 + __ffsll((unsigned long long)over) - 1);
    }
    if (lane) return;
    off[v + 1] = cnt;
    if (last + 1 > (int)__hip_atomic_load(info, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(info, (unsigned int)(last + 1));
}

// off[1 .. n] from counts to their running sum, off[0] = 0, info[2] = their sum;
// one workgroup.
__global__ __launch_bounds__(1024) void k_sparse_prefix(int *__restrict__ off, int n, unsigned int *__restrict__ info)
{
    __shared__ int wsum[16];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    int carry = 0;
    if (tid == 0) off[0] = 0;
    for (int i0 = 0; i0 < n; i0 += 1024) {
        const int i = i0 + tid;
        int x = i < n ? off[i + 1] : 0;
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(x, d, 64);
            if (lane >= d) x += o;
        }
        if (lane == 63) wsum[wv] = x;
        __syncthreads();
        int before = carry;
        for (int j = 0; j < 16; ++j) {
            before += j < wv ? wsum[j] : 0;
            carry += wsum[j];
        }
        if (i < n) off[i + 1] = before + x;
        __syncthreads();
    }
    if (tid == 0) info[2] = (unsigned int)carry;
}

__global__ __launch_bounds__(256) void k_sparse_fill(const uint32_t *__restrict__ y, int n, int stride,
                                                     const int *__restrict__ off, int *__restrict__ idx,
                                                     uint32_t *__restrict__ val)
{
    const int v = blockIdx.x * 4 + threadIdx.x / 64, lane = threadIdx.x & 63;
    if (v >= n) return;
    const uint32_t *row = y + (size_t)v * stride;
    int at = off[v];
    for (int i0 = 0; i0 < stride; i0 += 64) {
        const uint32_t t = i0 + lane < stride ? row[i0 + lane] : 0u;
        const uint64_t m = __ballot(t != 0);
        if (t) {
            const int o = at + __popcll(m & ((1ull << lane) - 1));
            idx[o] = i0 + lane;
            val[o] = t;
        }
        at += __popcll(m);
    }
}

int launch_sparse_count(const uint32_t *y, int n, int stride, int limit, int *off, unsigned int *info, hipStream_t st)
{
    if (n <= 0) return 0;
    if (launch_fill_i32((int *)info, 0, 1, st) || launch_fill_i32((int *)info + 1, -1, 1, st)) return -1;
    hipLaunchKernelGGL(k_sparse_count, dim3((unsigned)(n + 3) / 4), dim3(256), 0, st, y, n, stride, limit, off, info);
    hipLaunchKernelGGL(k_sparse_prefix, dim3(1), dim3(1024), 0, st, off, n, info);
    HIP_OK(hipGetLastError());
    return 0;
}

int launch_sparse_fill(const uint32_t *y, int n, int stride, const int *off, int *idx, uint32_t *val, hipStream_t st)
{
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_sparse_fill, dim3((unsigned)(n + 3) / 4), dim3(256), 0, st, y, n, stride, off, idx, val);
    HIP_OK(hipGetLastError());
    return 0;
}

// Position-weighted checksum of a word array: sum of (2i+1) * w_i (mod 2^64),
// so a moved, dropped or changed word changes it.  Grid-stride; one 64-bit
// atomic add per workgroup.
__global__ __launch_bounds__(256) void k_checksum(const uint32_t *__restrict__ w, size_t n,
                                                  unsigned long long *__restrict__ out)
{
    __shared__ unsigned long long part[256];
    unsigned long long acc = 0;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        acc += (2ull * i + 1ull) * (unsigned long long)w[i];
    part[threadIdx.x] = acc;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) part[threadIdx.x] += part[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(out, part[0]);
}

int launch_checksum(const uint32_t *w, size_t n, unsigned long long *out, hipStream_t st)
{
    if (n == 0) return 0;
    const size_t blocks = std::min<size_t>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(k_checksum, dim3((unsigned)blocks), dim3(256), 0, st, w, n, out);
    HIP_OK(hipGetLastError());
    return 0;
}

}  // namespace ipfe
