// k_sampler.hip -- discrete Gaussian sampling on gfx950, bit-exact with
// gaussian_sampler_S1_ori / S2_ori / S3 (src/gauss.c:705-785, :915-993,
// :1086-1163) on the AES-256-CTR stream of src/aes256ctr.c.
//
// The reference draws sample after sample from one sequential stream.  Each
// 384-byte refill ("chunk", 24 AES blocks) yields 8 candidates; a call takes
// accepted candidates in order until it has 4096, drops the rest of its last
// chunk, and the next call on the stream starts on the next chunk.  Here that
// becomes three data-parallel passes:
//   1. candidates: every chunk of a speculative window, in parallel: AES (LDS
//      T-tables), uniform/CDT/Bernoulli per candidate, wave ballot -> per-chunk
//      accept count and the accepted values compacted in order;
//   2. walk (k_gauss_walk.hip): counts into call boundaries; every chunk
//      labelled with (call, first output position);
//   3. scatter: every accepted candidate of a used chunk writes its three
//      residues to its call's polynomial.
#include <stdlib.h>

#include <algorithm>

#include "aes_dev.h"
#include "kernels.h"

namespace ipfe {

// Sampler constants (src/gauss.c:11-45): k per width, the Barrett factor
// floor(2^32/k), the uniform acceptance bound k*floor(2^32/k) and -1/k^2.
// Widths 1-3 are the reference's S1/S2/S3; 4 and 5 are the S2/S3 widths of the
// N = 2048 parameter set (the same algorithm with another k).
#define IPFE_SAMPLER_K {1ull, 266ull, 304214978ull, 608429953ull, 262147ull, 524287ull}
constexpr uint64_t kSamplerK[6] = IPFE_SAMPLER_K;
__constant__ uint64_t c_K[6] = IPFE_SAMPLER_K;
__constant__ uint64_t c_BF[6] = {0ull, (1ull << 32) / kSamplerK[1], (1ull << 32) / kSamplerK[2],
                                 (1ull << 32) / kSamplerK[3], (1ull << 32) / kSamplerK[4],
                                 (1ull << 32) / kSamplerK[5]};
__constant__ uint64_t c_UQ[6] = {0ull, kSamplerK[1] * ((1ull << 32) / kSamplerK[1]),
                                 kSamplerK[2] * ((1ull << 32) / kSamplerK[2]),
                                 kSamplerK[3] * ((1ull << 32) / kSamplerK[3]),
                                 kSamplerK[4] * ((1ull << 32) / kSamplerK[4]),
                                 kSamplerK[5] * ((1ull << 32) / kSamplerK[5])};
__constant__ double c_K2INV[6] = {0.0, -1.0 / (double)(long long)(kSamplerK[1] * kSamplerK[1]),
                                  -1.0 / (double)(long long)(kSamplerK[2] * kSamplerK[2]),
                                  -1.0 / (double)(long long)(kSamplerK[3] * kSamplerK[3]),
                                  -1.0 / (double)(long long)(kSamplerK[4] * kSamplerK[4]),
                                  -1.0 / (double)(long long)(kSamplerK[5] * kSamplerK[5])};

// Residue of a candidate on limb s of the stream's parameter set (src/gauss.c:773-779):
// mod_prime(z), then mod_prime(q - that) for a negative one.  No width's
// candidate reaches 2^34, below which one step of mod_prime's fold leaves 32
// bits on every modulus of the sets; q - m <= q needs no step.
__device__ __forceinline__ uint32_t stream_residue(const GaussStream *S, int s, uint64_t z, bool neg)
{
    const uint32_t q = S->q[s], a = S->fold[s] & 255u, b = S->fold[s] >> 8, lo = (1u << a) - 1;
    uint32_t m;
    if (z >> 34) {
        m = mod_prime_gen(z, q, a, b);
    } else {
        const uint32_t hi = (uint32_t)(z >> a), folded = ((uint32_t)z & lo) + (hi << b) - hi;
        m = z > 2 * q ? folded : (uint32_t)z;
        while (m > 2 * q) m = (m & lo) + ((m >> a) << b) - (m >> a);
        m = m >= q ? m - q : m;
    }
    if (neg) {
        m = q - m;
        m = m >= q ? m - q : m;
    }
    return m;
}

// CDT rows (low word, high word), src/gauss.c:62-72.
#define IPFE_CDT                                                                                            \
    {{2200310400551559144ull, 3327841033070651387ull}, {7912151619254726620ull, 380075531178589176ull},     \
     {5167367257772081627ull, 11604843442081400ull},   {5081592746475748971ull, 90134450315532ull},         \
     {6522074513864805092ull, 175786317361ull},        {2579734681240182346ull, 85801740ull},               \
     {8175784047440310133ull, 10472ull},               {2947787991558061753ull, 0ull},                      \
     {22489665999543ull, 0ull}}
constexpr uint64_t kCdt[9][2] = IPFE_CDT;
__constant__ uint64_t c_CDT[9][2] = IPFE_CDT;
// the upper halves of the high words that are not zero
constexpr uint32_t kCdtHigh[5] = {(uint32_t)(kCdt[0][1] >> 32), (uint32_t)(kCdt[1][1] >> 32),
                                  (uint32_t)(kCdt[2][1] >> 32), (uint32_t)(kCdt[3][1] >> 32),
                                  (uint32_t)(kCdt[4][1] >> 32)};
static_assert(kCdtHigh[4] > 0 && kCdt[5][1] >> 32 == 0, "five entries have an upper half");

// Coefficients of the 2^a polynomial, src/gauss.c:82-103 (IEEE-754 bit patterns).
__constant__ uint64_t c_EXP[10] = {0x3e833b70ffa2c5d4ull, 0x3eb4a480fda7e6e1ull, 0x3ef01b254493363full,
                                   0x3f242e0e0aa273ccull, 0x3f55d8a2334ed31bull, 0x3f83b2aa56db0f1aull,
                                   0x3fac6b08e11fc57eull, 0x3fcebfbdff556072ull, 0x3fe62e42fefa7fe6ull,
                                   0x3ff0000000000000ull};

extern const uint32_t *g_aes_te;  // device T-tables, set by the context

constexpr int CAND_THREADS = 256;
constexpr int CHUNK_WORDS = 96;

__device__ __forceinline__ int find_stream(const long long *prefix, int n, long long key)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (prefix[mid] <= key) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// Bernoulli decision (src/gauss.c:204-264 and the S2/S3 copies): the
// reference's exact sequence of IEEE double operations and integer bit tricks.
// rb points at the 36 Bernoulli bytes of the candidate's group.
// bernoulli_exp: the bits the uniform word is compared with.
__device__ __forceinline__ uint64_t bernoulli_exp(uint64_t b, double k2inv)
{
    double vx = __longlong_as_double((long long)(b | 0x4330000000000000ull)) - 4503599627370496.0;
    vx = __dmul_rn(vx, k2inv);
    double fl = floor(vx);
    double sh = __dadd_rn(fl, 6755399441055744.0);
    uint64_t t = ((uint64_t)__double_as_longlong(sh) - 0x4338000000000000ull) << 52;
    double a = __dsub_rn(vx, fl);
    double s = __fma_rn(__longlong_as_double((long long)c_EXP[0]), a, __longlong_as_double((long long)c_EXP[1]));
#pragma unroll
    for (int i = 2; i < 10; ++i) s = __fma_rn(s, a, __longlong_as_double((long long)c_EXP[i]));
    return t + (uint64_t)__double_as_longlong(s);
}

__device__ __forceinline__ bool bernoulli_bit(uint64_t b, double k2inv, const uint32_t *rb, int ln)
{
    const uint64_t res = bernoulli_exp(b, k2inv);
    uint64_t res_mant = (res & ((1ull << 52) - 1)) | (1ull << 52);
    uint64_t e = (res >> 52) + (uint64_t)(long long)-1003;
    uint64_t res_exp = (e < 64) ? (1ull << e) : 0ull;
    uint64_t rm = ((uint64_t)rb[2 * ln + 1] << 32) | rb[2 * ln];
    uint64_t r_exp = (rm >> 53) | ((uint64_t)((rb[8] >> (8 * ln)) & 255u) << 11);
    uint64_t r_mant = rm & ((1ull << 53) - 1);
    uint64_t bits = (r_mant - res_mant) & (r_exp - res_exp);
    return (bits >> 63) != 0 || res == 0x3FF0000000000000ull;
}

// One candidate of a chunk held in LDS (96 little-endian words).  Lanes 8t..8t+7
// of a wave evaluate candidates 0..7 of one chunk together: the uniform words
// are shared through ballots, so every lane of the wave must call this.
struct Cand {
    uint64_t z;
    uint32_t sgn;
    bool acc;
};

// AES blocks of a chunk k_gauss_firsts computes by default: 0..15 (bytes 0..255) and 17
// (bytes 272..287, holding the sign byte 280).  Candidates read bytes 0..199
// (CDT and Bernoulli words), the uniform words from byte 200 and byte 280; the
// uniform scan stays below byte 256 unless it needs more than 14 words (seven
// or more rejections, about 1e-11 per chunk).  Such a chunk sets status bit 4
// and the caller reruns the group with all 24 blocks.
constexpr int PART_BLOCKS = 17;
__device__ __forceinline__ int chunk_block(int j, int full) { return (full || j < 16) ? j : 17; }

// ulim: uniform words a partial chunk may scan (14 covers its blocks; lower
// values exist to exercise the rerun).
__device__ __forceinline__ Cand eval_candidate(const uint32_t *ch, int c, int which, bool valid, int *status,
                                               int full, int ulim)
{
    const uint64_t K = c_K[which], BF = c_BF[which];
    const uint32_t UQ = (uint32_t)c_UQ[which];
    const double K2INV = c_K2INV[which];
    const int sh = (threadIdx.x & 63) & 56;
    // uniform_sampler (src/gauss.c:609-703): the c-th word below UQ from byte 200 on
    const uint32_t w0 = ch[50 + c], w1 = ch[58 + c], w2 = ch[66 + c];
    const uint64_t m0 = __ballot(w0 < UQ), m1 = __ballot(w1 < UQ), m2 = __ballot(w2 < UQ);
    const uint32_t mask = (uint32_t)((m0 >> sh) & 0xffu) | ((uint32_t)((m1 >> sh) & 0xffu) << 8) |
                          ((uint32_t)((m2 >> sh) & 0xffu) << 16);
    int pos = c;
    if ((mask & 0xffu) != 0xffu) {
        int seen = 0;
        bool partial_miss = false;
        pos = -1;
        for (int u = 0; u < 46; ++u) {
            if (!full && u >= ulim) {
                partial_miss = true;  // word 64 on lies in a block not computed
                break;
            }
            const bool kept = (u < 24) ? ((mask >> u) & 1u) : (ch[50 + u] < UQ);
            if (kept) {
                if (seen == c) { pos = u; break; }
                ++seen;
            }
        }
        if (pos < 0) {
            if (valid) atomicOr(status, partial_miss ? 4 : 2);
            pos = 0;
        }
    }
    const uint64_t w = ch[50 + pos];
    uint64_t y = w - ((((w * BF) >> 32) + 1) * K);
    y = y + (y >> 63) * K;

    // cdt_sampler (src/gauss.c:122-154)
    const int g = c >> 2, ln = c & 3;
    const uint32_t *gb = ch + 25 * g;
    const uint64_t r1 = (((uint64_t)gb[2 * ln + 1] << 32) | gb[2 * ln]) & 0x7fffffffffffffffull;
    const uint64_t r2 = (((uint64_t)gb[8 + 2 * ln + 1] << 32) | gb[8 + 2 * ln]) & 0x7fffffffffffffffull;
    uint32_t xs = 0;
#pragma unroll
    for (int i = 0; i < 9; ++i) xs += (r2 < c_CDT[i][1]) | ((r2 == c_CDT[i][1]) & (r1 < c_CDT[i][0]));

    const uint64_t xk = (uint64_t)xs * (uint64_t)(uint32_t)K;
    Cand out;
    out.z = xk + y;
    const uint64_t bin = (uint64_t)(uint32_t)(out.z + xk) * (uint64_t)(uint32_t)y;
    const bool bit = bernoulli_bit(bin, K2INV, gb + 16, ln);
    out.sgn = (ch[70] >> c) & 1u;  // sign byte 280
    out.acc = bit && (out.z != 0 || out.sgn != 0);
    return out;
}

// ---------------------------------------------------------------------------
// Candidate pass.
//
// What a chunk's eight candidates read (byte offsets in the 384-byte chunk;
// candidate c = 4 g + ln): the CDT words r1, r2 at 100 g + 8 ln and 32 beyond,
// the Bernoulli words at 100 g + 64 + 8 ln and the byte 100 g + 96 + ln, the
// uniform words from byte 200, the sign byte 280.  r1 decides only where r2
// equals a CDT entry's high word, so blocks 0, 1 and 7 (r1 alone) and block 15
// (the uniform words past the tenth) are not computed; nor is more than the
// high 32 bits of r2 and of the Bernoulli word looked at, whose low halves
// decide only where the high halves tie.  That leaves the 12 blocks 2..6, 8..14
// of 24 a chunk -- and block 17, the sign, for streams whose values are stored --
// where all words of blocks 0..15 took 16 (17).  What that leaves open is looked
// at by the candidate's lane with the block it needs: the next uniform words
// after a third rejected one among ten (7e-5 of chunks), the sign of a zero
// candidate of a stream that stores no values (0.2% of S1's), the whole words
// after a tie (6 in 2^31, 1 in 2^21).  A lane's blocks go through the tile's
// windows and scalar round keys as the others' do: 1 call of S1 13.6 us, 64 of S2
// and S3 32 and 35, 500 streams of 3 S1 calls 275 (with every open candidate
// recomputed from up to nine whole blocks, each from the first round: 68, 60, 71
// and 641; the kernel for all words 15, 42, 55 and 560).
//
// Each wave works alone: 16 chunks are 192 blocks, three full rounds of the
// wave (blocks 2-5, 8-11 and 6, 12-14, so that a round's lanes need the same
// output words: two of four in the first two), then 128 candidates, two full
// rounds.  No workgroup barriers, so the lookups of some waves run under the
// arithmetic of others.  The 28 words a chunk leaves for its candidates fit 16
// waves' buffers beside 128 KiB of tables.
//
// Bound by the LDS lookups (197 a block, 64 lanes in 2 CU cycles) and the VALU,
// about equally: 5.8 G chunks/s on the
// streams of 2,048 rows of 124 slots (58 ms; 114 ms for all words of blocks 0..15
// in 512-thread workgroups with T0 and T2 alone, encryption and evaluation
// alternating across barriers).
//
// Words of a chunk in the wave's buffer (28, 112 bytes):
//    0..3  r2 high of candidates 0..3       4..7  their Bernoulli high words
//    8     bytes of candidates 0..3         9..12 r2 high of 4..7
//   13..16 Bernoulli high words of 4..7    17     their bytes
//   18..27 uniform words 0..9
// ---------------------------------------------------------------------------
typedef const __attribute__((address_space(4))) uint32_t *RoundKeys;  // scalar loads

// TM: the T-table layout in LDS -- 0: four 1 KiB tables; 1: T0 replicated per
// bank (AesTabRep); 2: T0 and T2 (AesTabRep2); 3: all four (AesTabRep4).
template <int TM>
struct AesLayout;
template <>
struct AesLayout<0> {
    using Tab = AesTab4;
    static constexpr int words = AES_TABLE_WORDS;
    static __device__ void stage(uint32_t *te, const uint32_t *g) { aes_stage_tables(te, g); }
};
template <>
struct AesLayout<1> {
    using Tab = AesTabRep;
    static constexpr int words = AES_REP_WORDS;
    static __device__ void stage(uint32_t *te, const uint32_t *g) { aes_stage_tables_rep(te, g); }
};
template <>
struct AesLayout<2> {
    using Tab = AesTabRep2;
    static constexpr int words = AES_REP2_WORDS;
    static __device__ void stage(uint32_t *te, const uint32_t *g) { aes_stage_tables_rep2(te, g); }
};
template <>
struct AesLayout<3> {
    using Tab = AesTabRep4;
    static constexpr int words = AES_REP4_WORDS;
    static __device__ void stage(uint32_t *te, const uint32_t *g) { aes_stage_tables_rep4(te, g); }
};

constexpr int CAND_NT = 1024, CAND_WAVES = CAND_NT / 64;
constexpr int SUB_CHUNKS = 16, SUB_WORDS = 28, TILE_CHUNKS = 64;
constexpr int CAND_WINDOWS = 8;  // of 256 counters: a 64-chunk tile's 1,536 touch at most seven
static_assert(SUB_CHUNKS * SUB_WORDS + 8 * CAND_WINDOWS == 512, "the wave's buffer");

// The parameters of a sampler width and the arithmetic all candidates share.
struct WidthConsts {
    uint32_t K, BF, UQ;
    double k2inv;
    __device__ explicit WidthConsts(int which)
        : K((uint32_t)c_K[which]), BF((uint32_t)c_BF[which]), UQ((uint32_t)c_UQ[which]), k2inv(c_K2INV[which])
    {
    }
};

// uniform word -> y (src/gauss.c:609-703): y = w - (floor(w BF / 2^32) + 1) K,
// plus K when that is negative.
__device__ __forceinline__ uint32_t uniform_y(uint32_t w, const WidthConsts &wc)
{
    const uint32_t r = w - __umulhi(w, wc.BF) * wc.K;
    return r >= wc.K ? r - wc.K : r;
}

// z = xs K + y and the bits of 2^a that the Bernoulli step compares with
// (bernoulli_bit above, the reference's IEEE double sequence).
__device__ __forceinline__ uint64_t cand_exp(uint32_t xs, uint32_t y, const WidthConsts &wc, uint64_t &z)
{
    const uint64_t xk = (uint64_t)xs * wc.K;
    z = xk + y;
    const uint64_t b = (uint64_t)(uint32_t)(z + xk) * y;
    return bernoulli_exp(b, wc.k2inv);
}

// r_exp < res_exp: r_exp the 19 bits above the Bernoulli word's 53, res_exp =
// 2^e with e from the exponent field (0 past 63)
__device__ __forceinline__ bool bernoulli_exp_less(uint32_t res_hi, uint32_t rm_hi, uint32_t byte)
{
    const uint32_t e = (res_hi >> 20) - 1003u, r_exp = (rm_hi >> 21) | byte << 11;
    return e < 64u && (r_exp >> min(e, 31u)) == 0;
}

// One candidate from whole words of its chunk, for the lanes whose candidate the
// high words leave open; y of its uniform word, block(b, o): AES block b of
// the chunk.
template <class Block>
__device__ Cand cand_whole(const Block &block, int c, uint32_t y, const WidthConsts &wc, bool lazy_sign)
{
    const int g = c >> 2, ln = c & 3;
    uint32_t o[4] = {0, 0, 0, 0};
    int cur = -1;
    uint32_t w[8];  // r1, r2, Bernoulli (low, high each), byte word, sign
    const int at[8] = {25 * g + 2 * ln,      25 * g + 2 * ln + 1,  25 * g + 8 + 2 * ln, 25 * g + 9 + 2 * ln,
                       25 * g + 16 + 2 * ln, 25 * g + 17 + 2 * ln, 25 * g + 24,         70};
#pragma unroll 1
    for (int j = 0; j < 8; ++j) {
        int i = at[0];
#pragma unroll
        for (int v = 1; v < 8; ++v) i = j == v ? at[v] : i;
        if (cur != i >> 2) {
            cur = i >> 2;
            block(cur, o);
        }
        const uint32_t lo = (i & 1) ? o[1] : o[0], hi = (i & 1) ? o[3] : o[2], t = (i & 2) ? hi : lo;
#pragma unroll
        for (int v = 0; v < 8; ++v) w[v] = j == v ? t : w[v];
    }
    const uint64_t r1 = (((uint64_t)w[1] << 32) | w[0]) & 0x7fffffffffffffffull;
    const uint64_t r2 = (((uint64_t)w[3] << 32) | w[2]) & 0x7fffffffffffffffull;
    uint32_t xs = 0;
#pragma unroll
    for (int i = 0; i < 9; ++i) xs += (r2 < c_CDT[i][1]) | ((r2 == c_CDT[i][1]) & (r1 < c_CDT[i][0]));
    Cand out;
    const uint64_t res = cand_exp(xs, y, wc, out.z);
    const uint64_t rm = ((uint64_t)w[5] << 32) | w[4];
    const uint64_t res_mant = (res & ((1ull << 52) - 1)) | (1ull << 52), r_mant = rm & ((1ull << 53) - 1);
    const bool bit = (r_mant < res_mant && bernoulli_exp_less((uint32_t)(res >> 32), w[5], (w[6] >> (8 * ln)) & 255u)) ||
                     res == 0x3FF0000000000000ull;
    out.sgn = (!lazy_sign || out.z == 0) ? (w[7] >> c) & 1u : 0u;
    out.acc = bit && (out.z != 0 || out.sgn != 0);
    return out;
}

template <int TM>
__global__ __launch_bounds__(CAND_NT) void k_gauss_candidates(const GaussStream *__restrict__ streams, int nstreams,
                                                               const long long *__restrict__ chunk_prefix,
                                                               long long nchunks_total,
                                                               const uint32_t *__restrict__ te_global,
                                                               uint8_t *__restrict__ cnt, uint64_t *__restrict__ vals,
                                                               int *__restrict__ status, int full, int ulim, int whole)
{
    using Tab = typename AesLayout<TM>::Tab;
    __shared__ __align__(16) uint32_t te[AesLayout<TM>::words];
    __shared__ __align__(16) uint32_t bufs[CAND_WAVES][512];
    AesLayout<TM>::stage(te, te_global);
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // This wave's run of groups of 16 chunks, taken in tiles of up to four groups
    // within a stream (one window pass and, for stored values, one round of sign
    // blocks a tile: 64 chunks fill its lanes).  Runs end on any group: dealt in
    // whole tiles of one size, a plan of a few tiles a wave left most waves
    // idle in its last round (full streams of S3, 800 calls: 305 -> 280 us, 126: 93
    // -> 85).  The first waves of all workgroups come first: fewer groups than waves
    // spread over all CUs (4 calls: 22 -> 14 us), and a plan's full streams, whose
    // chunks cost more, over many (all in a few workgroups they made 2,048 rows 7%
    // slower).
    const long long groups = nchunks_total / SUB_CHUNKS;
    const long long waves = min((long long)gridDim.x * CAND_WAVES, groups), me = (long long)wv * gridDim.x + blockIdx.x;
    if (me >= waves) return;
    const long long t0 = me * groups / waves * SUB_CHUNKS, t1 = (me + 1) * groups / waves * SUB_CHUNKS;
    const Tab tb(te);
    uint32_t *buf = bufs[wv], *win = buf + SUB_CHUNKS * SUB_WORDS;
    int si = __builtin_amdgcn_readfirstlane(find_stream(chunk_prefix, nstreams, t0));
    auto wave_sync = [] {  // the wave's LDS accesses stay in order across this point
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
    };
    for (long long t = t0; t < t1;) {  // the run's part of each stream it meets
        while (si + 1 < nstreams && chunk_prefix[si + 1] <= t) ++si;
        const GaussStream *S = streams + si;
        const long long stream0 = chunk_prefix[si];
        const long long t_next = si + 1 < nstreams ? min(t1, chunk_prefix[si + 1]) : t1;
        const int chunk_first = (int)(t - stream0), chunk_end = min((int)(t_next - stream0), S->nchunks);
        t = t_next;
        const WidthConsts wc(S->which);
        const bool store_vals = !S->coef0_only;
        const uint32_t nonce = S->nonce;
        const uint64_t rk_addr = reinterpret_cast<uint64_t>(&S->rk[0]);
        // The round keys are read anew for every round of blocks (the empty
        // asm keeps the loads there): 64 scalar registers held across the
        // evaluation would be spilled to vector lanes.
        auto keys = [rk_addr]() {
            uint64_t a = rk_addr;
            asm volatile("" : "+s"(a));
            return (RoundKeys)a;
        };
        for (int chunk0 = chunk_first; chunk0 < chunk_end; chunk0 += TILE_CHUNKS) {
            const int nch = min(TILE_CHUNKS, chunk_end - chunk0);
            // windows of 256 counters the tile touches (counters wrap at 2^32)
            const uint32_t c_lo = (uint32_t)chunk0 * 24u, w0 = c_lo >> 8;
            const int nw = (int)(((c_lo & 255u) + (uint32_t)(nch * 24 - 1)) >> 8) + 1;
            wave_sync();
            if (lane < nw) aes256_ctr_window(tb, keys(), nonce, (w0 + lane) & 0xffffffu, win + 8 * lane);
            wave_sync();
            auto window = [&](uint32_t ctr) { return win + 8 * (((ctr >> 8) - w0) & (CAND_WINDOWS - 1)); };
            uint32_t sign = 0;  // lane l: the sign word of the tile's chunk l
            if (store_vals) {
                const uint32_t ctr = (uint32_t)(chunk0 + min(lane, nch - 1)) * 24u + 17u;
                uint32_t o[4];
                const RoundKeys rk = keys();
                aes256_ctr_block_win<4>(tb, rk, rk + 60, window(ctr), ctr, o);
                sign = o[2];
            }
            for (int s = 0; s < nch; s += SUB_CHUNKS) {
                const int nsub = min(SUB_CHUNKS, nch - s);
                {
                    const int k = lane >> 2, j = lane & 3;
                    const uint32_t base = (uint32_t)(chunk0 + s + min(k, nsub - 1)) * 24u;
                    uint32_t *d = buf + SUB_WORDS * k;
                    uint32_t o[4];
                    {
                        const uint32_t ctr = base + 2 + j;
                        const RoundKeys rk = keys();
                        aes256_ctr_block_win<2 | 8>(tb, rk, rk + 60, window(ctr), ctr, o);
                        *reinterpret_cast<uint2 *>(d + 2 * j) = make_uint2(o[1], o[3]);
                    }
                    {
                        const uint32_t ctr = base + 8 + j;
                        const RoundKeys rk = keys();
                        aes256_ctr_block_win<1 | 4>(tb, rk, rk + 60, window(ctr), ctr, o);
                        *reinterpret_cast<uint2 *>(d + 8 + 2 * j) = make_uint2(o[0], o[2]);
                    }
                    {
                        const uint32_t ctr = base + (j == 0 ? 6 : 11 + j);
                        const RoundKeys rk = keys();
                        aes256_ctr_block_win(tb, rk, rk + 60, window(ctr), ctr, o);
                        if (j == 0)
                            d[8] = o[0];  // over block 8's first word, which no candidate reads
                        else
                            *reinterpret_cast<uint4 *>(d + 12 + 4 * j) = make_uint4(o[0], o[1], o[2], o[3]);
                    }
                }
                wave_sync();
    #pragma unroll 1
                for (int e = 0; e < 2; ++e) {
                    const int k = 8 * e + (lane >> 3), c = lane & 7, sh = lane & 56;
                    const bool valid = k < nsub;
                    const uint32_t *q = buf + SUB_WORDS * k;
                    // a block of the lane's chunk beyond the ones in the buffer
                    auto block = [&](int b, uint32_t (&o)[4]) {
                        const uint32_t ctr = (uint32_t)(chunk0 + s + k) * 24u + b;
                        const RoundKeys rk = keys();
                        aes256_ctr_block_win(tb, rk, rk + 60, window(ctr), ctr, o);
                    };
                    // the c-th uniform word below UQ
                    uint32_t w = q[18 + c];
                    const uint64_t kept = __ballot(w < wc.UQ);
                    if (kept != ~0ull) {
                        const uint32_t bad = ~((uint32_t)((kept >> sh) & 0xffu) | (q[26] < wc.UQ ? 256u : 0u) |
                                               (q[27] < wc.UQ ? 512u : 0u));
                        // its position: c plus the rejected words up to it
                        int pos = c;
    #pragma unroll
                        for (int it = 0; it < 3; ++it) pos = c + __popc(bad & ((2u << min(pos, 15)) - 1u));
                        const bool far = pos >= min(ulim, 10) || pos != c + __popc(bad & ((2u << min(pos, 15)) - 1u));
                        w = q[18 + min(pos, 9)];
                        if (far && valid) {  // past the tenth word, after a chain of rejections or past the limit
                            uint32_t o[4];
                            int seen = 0, u = 0;
                            const int end = full ? 46 : ulim;
                            for (; u < end; ++u) {
                                uint32_t t = q[18 + min(u, 9)];
                                if (u >= 10) {
                                    const int i = 50 + u;
                                    if ((i & 3) == 0) block(i >> 2, o);
                                    const uint32_t lo = (i & 1) ? o[1] : o[0], hi = (i & 1) ? o[3] : o[2];
                                    t = (i & 2) ? hi : lo;
                                }
                                if (t < wc.UQ && seen++ == c) {
                                    w = t;
                                    break;
                                }
                            }
                            if (u == end) atomicOr(status, full ? 2 : 4);
                        }
                    }
                    const uint32_t y = uniform_y(w, wc);
                    // CDT rank by the high word
                    const uint32_t r2h = q[c < 4 ? c : c + 5] & 0x7fffffffu;
                    uint32_t xs = 0;
                    bool tie = r2h == 0;  // the entries from the sixth on have a zero high word
    #pragma unroll
                    for (int i = 0; i < 5; ++i) {
                        xs += r2h < kCdtHigh[i];
                        tie = tie || r2h == kCdtHigh[i];
                    }
                    Cand cd;
                    const uint64_t res = cand_exp(xs, y, wc, cd.z);
                    const uint32_t rm_hi = q[c < 4 ? 4 + c : 9 + c], bytes = q[c < 4 ? 8 : 17];
                    const uint32_t res_hi = (uint32_t)(res >> 32);
                    const uint32_t mant = (res_hi & 0xfffffu) | 0x100000u, rmant = rm_hi & 0x1fffffu;
                    const bool bit = (rmant < mant && bernoulli_exp_less(res_hi, rm_hi, (bytes >> (8 * (c & 3))) & 255u)) ||
                                     res == 0x3FF0000000000000ull;
                    cd.sgn = store_vals ? (__shfl(sign, s + k, 64) >> c) & 1u : 0u;
                    cd.acc = valid && bit && (store_vals ? (cd.z != 0 || cd.sgn != 0) : true);
                    if (valid && (whole || tie || rmant == mant)) {
                        cd = cand_whole(block, c, y, wc, !store_vals);
                    } else if (!store_vals && cd.acc && cd.z == 0) {  // accepted if its sign is set
                        uint32_t o[4];
                        block(17, o);
                        cd.acc = (o[2] >> c) & 1u;
                    }
                    const uint64_t am = __ballot(cd.acc);
                    const uint32_t gm = (uint32_t)((am >> sh) & 0xffu);
                    if (valid) {
                        const long long gc = S->chunk_base + chunk0 + s + k;
                        if (c == 0) cnt[gc] = (uint8_t)__popc(gm);
                        if (store_vals && cd.acc)
                            vals[gc * 8 + __popc(gm & ((1u << c) - 1u))] = cd.z | ((uint64_t)cd.sgn << 63);
                    }
                }
                wave_sync();
            }
        }
    }
}

// Compact streams: sample 0 of every call.  Item t (a call of a compact
// stream) has its first non-empty chunk in firsts[t]; the chunk is recomputed
// and its first accepted candidate written as 3 residues at out0 + 3 call.
constexpr int FIRST_TILE = 32;

__global__ __launch_bounds__(CAND_THREADS) void k_gauss_firsts(const GaussStream *__restrict__ streams, int nstreams,
                                                                const long long *__restrict__ first_prefix,
                                                                const long long *__restrict__ firsts, long long nitems,
                                                                const uint32_t *__restrict__ te_global,
                                                                int *__restrict__ status, int full, int ulim)
{
    __shared__ uint32_t te[AES_TABLE_WORDS];
    __shared__ uint32_t ks[FIRST_TILE * CHUNK_WORDS];
    __shared__ int s_stream[FIRST_TILE];
    __shared__ long long s_chunk[FIRST_TILE];
    aes_stage_tables(te, te_global);
    const long long t0 = (long long)blockIdx.x * FIRST_TILE;
    if (threadIdx.x < FIRST_TILE) {
        const long long t = t0 + threadIdx.x;
        int si = -1;
        long long ch = 0;
        if (t < nitems) {
            si = find_stream(first_prefix, nstreams, t);
            ch = firsts[t] - streams[si].chunk_base;
        }
        s_stream[threadIdx.x] = si;
        s_chunk[threadIdx.x] = ch;
    }
    __syncthreads();
    // AES: 24 blocks per item, each item possibly from a different stream
    const int nb = full ? 24 : PART_BLOCKS;
    for (int g = threadIdx.x; g < FIRST_TILE * nb; g += CAND_THREADS) {
        const int k = g / nb, blk = chunk_block(g - nb * k, full);
        const int si = s_stream[k];
        if (si < 0) continue;
        const GaussStream *S = streams + si;
        uint32_t o[4];
        aes256_ctr_block(S->rk, te, S->nonce, (uint32_t)(s_chunk[k] * 24 + blk), o);
        uint32_t *d = ks + k * CHUNK_WORDS + blk * 4;
        d[0] = o[0]; d[1] = o[1]; d[2] = o[2]; d[3] = o[3];
    }
    __syncthreads();
    const int sh = (threadIdx.x & 63) & 56;
    const int k = threadIdx.x >> 3, c = threadIdx.x & 7;  // 32 items x 8 candidates = 256 threads
    const int si = s_stream[k];
    const bool valid = si >= 0;
    const int which = valid ? streams[si].which : 1;
    const Cand cd = eval_candidate(ks + k * CHUNK_WORDS, c, which, valid, status, full, ulim);
    const uint64_t am = __ballot(cd.acc && valid);
    const uint32_t gm = (uint32_t)((am >> sh) & 0xffu);
    if (valid && cd.acc && (gm & ((1u << c) - 1u)) == 0) {
        const GaussStream *S = streams + si;
        const long long call = t0 + k - first_prefix[si];
        uint32_t *out = S->out0 + (long long)S->nmod * call;
        for (int s = 0; s < S->nmod; ++s) out[s] = stream_residue(S, s, cd.z, cd.sgn != 0);
    }
}

// Accepted values of full streams to their output residues.  A wave takes
// SCATTER_CHUNKS consecutive chunks, 16 at a time with 4 lanes a chunk and two
// values a lane: streams start on a multiple of 16 chunks, so the 16 share a
// stream, found once a wave and followed from there, and all their loads are
// issued before any is used.  10,240 calls of S3 on 1,024 streams: 460 us (844
// with 8 lanes a chunk, 8 chunks and a search of the stream a wave, which waited
// on one chain of loads after another), 800 on two streams 32 (42): about 106 B
// read and written a chunk at 3.2 TB/s.  16 chunks a wave 530 and 30, 64 470 and
// 38, 128 504 and 50; stores past the caches 735.
constexpr int SCATTER_CHUNKS = 32;

__global__ __launch_bounds__(256) void k_gauss_scatter(const GaussStream *__restrict__ streams, int nstreams,
                                                      const long long *__restrict__ chunk_prefix,
                                                      long long nchunks_total, const uint8_t *__restrict__ cnt,
                                                      const uint64_t *__restrict__ vals, const int *__restrict__ pos)
{
    constexpr int G = SCATTER_CHUNKS / 16;
    const int lane = threadIdx.x & 63, slot = 2 * (lane & 3);
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (long long base = ((long long)blockIdx.x * 4 + wv) * SCATTER_CHUNKS; base < nchunks_total;
         base += (long long)gridDim.x * 4 * SCATTER_CHUNKS) {
        int info[G], n[G];
        ulonglong2 v[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            info[g] = -1;
            if (base + 16 * g >= nchunks_total) continue;  // nchunks_total is a multiple of 16
            const long long gc = base + 16 * g + (lane >> 2);
            info[g] = pos[gc];
            n[g] = cnt[gc];
            v[g] = *reinterpret_cast<const ulonglong2 *>(vals + gc * 8 + slot);
        }
        int si = __builtin_amdgcn_readfirstlane(find_stream(chunk_prefix, nstreams, base));
#pragma unroll
        for (int g = 0; g < G; ++g) {
            while (si + 1 < nstreams && chunk_prefix[si + 1] <= base + 16 * g) ++si;
            if (info[g] < 0) continue;
            const GaussStream *S = streams + si;
            const int call = info[g] >> 13, off = (info[g] & 0x1fff) + slot;
            // output residues (src/gauss.c:773-779)
            uint32_t *out = ((call == 0) ? S->out0 : S->out1 + (long long)(call - 1) * S->out_stride) + off;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                if (slot + j >= n[g] || off + j >= S->slen) continue;
                const uint64_t w = j ? v[g].y : v[g].x, z = w & 0x7fffffffffffffffull;
                for (int s = 0; s < S->nmod; ++s)
                    out[(long long)s * S->slen + j] = stream_residue(S, s, z, (w >> 63) != 0);
            }
        }
    }
}

__global__ void k_fill_i32(int *p, int v, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

// sample_polya (src/sample.c:56-128): coefficient i = LE64(keystream[8i..8i+8))
// mod q_j, keystream of AES-256-CTR(seed, nonce 0) from counter 0.  Any
// parameter set: n coefficients on nmod limbs, a [nmod][n].
struct PolyaArgs {
    int n, nmod;
    uint32_t q[4];
};
__global__ void k_sample_polya(const uint32_t *__restrict__ rk, const uint32_t *__restrict__ te_global,
                               uint32_t *__restrict__ a, PolyaArgs pa)
{
    __shared__ uint32_t te[AES_TABLE_WORDS];
    aes_stage_tables(te, te_global);
    __syncthreads();
    const uint32_t blk = blockIdx.x * blockDim.x + threadIdx.x;  // n / 2 blocks
    if (blk >= (uint32_t)pa.n / 2) return;
    uint32_t o[4];
    aes256_ctr_block(rk, te, 0u, blk, o);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint64_t v = ((uint64_t)o[2 * h + 1] << 32) | o[2 * h];
        const uint32_t i = 2 * blk + h;
        for (int s = 0; s < pa.nmod; ++s) a[(size_t)s * pa.n + i] = (uint32_t)(v % pa.q[s]);
    }
}

__global__ void k_aes_ctr(const uint32_t *__restrict__ rk, const uint32_t *__restrict__ te_global, uint32_t nonce,
                          uint32_t ctr0, uint32_t nblocks, uint32_t *__restrict__ out)
{
    __shared__ uint32_t te[AES_TABLE_WORDS];
    aes_stage_tables(te, te_global);
    __syncthreads();
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nblocks) return;
    uint32_t o[4];
    aes256_ctr_block(rk, te, nonce, ctr0 + b, o);
    out[4 * b + 0] = o[0]; out[4 * b + 1] = o[1]; out[4 * b + 2] = o[2]; out[4 * b + 3] = o[3];
}

// ---------------------------------------------------------------------------
// CUFE_AES_REP: the table layout of the candidate pass -- 0: the four 1 KiB
// T-tables; 1, 2: T0 replicated; 3: T0 and T2; else (default) all four.
static int aes_rep_mode()
{
    const char *e = getenv("CUFE_AES_REP");
    return e && *e ? atoi(e) : 4;
}

// Uniform words a partial chunk may scan before it asks for all 24 blocks:
// 14 (all its blocks hold); CUFE_GAUSS_SCAN in [8, 14] lowers it so tests can
// drive the rerun path.
static int scan_limit()
{
    const char *e = getenv("CUFE_GAUSS_SCAN");
    const int v = e && *e ? atoi(e) : 14;
    return v < 8 ? 8 : (v > 14 ? 14 : v);
}

// One workgroup per CU: its tables and buffers take the whole LDS.
static int candidate_blocks()
{
    static const int cus = [] {
        hipDeviceProp_t prop;
        int d = 0;
        if (hipGetDevice(&d) != hipSuccess || hipGetDeviceProperties(&prop, d) != hipSuccess) return 256;
        return prop.multiProcessorCount;
    }();
    return cus;
}

int launch_gauss_candidates(const GaussStream *d_streams, int nstreams, const long long *d_chunk_prefix,
                            long long nchunks_total, uint8_t *cnt, uint64_t *vals, int *status, int full,
                            hipStream_t st)
{
    if (nchunks_total <= 0) return 0;
    if (nchunks_total % SUB_CHUNKS) {
        ipfe_set_error("Gaussian candidates: %lld chunks, not a multiple of 16", nchunks_total);
        return -1;
    }
    const unsigned grid = (unsigned)std::min<long long>(nchunks_total / SUB_CHUNKS, candidate_blocks());
    const int rep = aes_rep_mode();
    // CUFE_GAUSS_WHOLE=1 (tests): every candidate from whole words
    const char *w = getenv("CUFE_GAUSS_WHOLE");
    const int whole = w && atoi(w) != 0;
#define CAND(TM)                                                                                                   \
    hipLaunchKernelGGL(k_gauss_candidates<TM>, dim3(grid), dim3(CAND_NT), 0, st, d_streams, nstreams, d_chunk_prefix, \
                       nchunks_total, g_aes_te, cnt, vals, status, full, scan_limit(), whole)
    if (rep >= 4)
        CAND(3);
    else if (rep == 3)
        CAND(2);
    else if (rep >= 1)
        CAND(1);
    else
        CAND(0);
#undef CAND
    HIP_OK(hipGetLastError());
    return 0;
}

int launch_gauss_scatter(const GaussStream *d_streams, int nstreams, const long long *d_chunk_prefix,
                         long long nchunks_total, const uint8_t *cnt, const uint64_t *vals, const int *pos,
                         hipStream_t st)
{
    if (nchunks_total <= 0) return 0;
    if (nchunks_total % 16) {
        ipfe_set_error("Gaussian scatter: %lld chunks, not a multiple of 16", nchunks_total);
        return -1;
    }
    constexpr int per_wg = 4 * SCATTER_CHUNKS;
    const unsigned grid = (unsigned)std::min<long long>((nchunks_total + per_wg - 1) / per_wg, 1ll << 20);
    hipLaunchKernelGGL(k_gauss_scatter, dim3(grid), dim3(256), 0, st, d_streams, nstreams, d_chunk_prefix,
                       nchunks_total, cnt, vals, pos);
    HIP_OK(hipGetLastError());
    return 0;
}

int launch_gauss_firsts(const GaussStream *d_streams, int nstreams, const long long *d_first_prefix,
                        const long long *firsts, long long nitems, int *status, int full, hipStream_t st)
{
    if (nitems <= 0) return 0;
    hipLaunchKernelGGL(k_gauss_firsts, dim3((unsigned)((nitems + FIRST_TILE - 1) / FIRST_TILE)), dim3(CAND_THREADS), 0,
                       st, d_streams, nstreams, d_first_prefix, firsts, nitems, g_aes_te, status, full, scan_limit());
    HIP_OK(hipGetLastError());
    return 0;
}

int launch_fill_i32(int *p, int v, size_t n, hipStream_t st)
{
    if (n == 0) return 0;
    const unsigned grid = (unsigned)std::min<size_t>((n + 255) / 256, (size_t)1 << 20);
    hipLaunchKernelGGL(k_fill_i32, dim3(grid), dim3(256), 0, st, p, v, n);
    HIP_OK(hipGetLastError());
    return 0;
}

int launch_sample_polya(const uint32_t *d_rk, uint32_t *a, hipStream_t st)
{
    const uint32_t q[3] = {qmod(0), qmod(1), qmod(2)};
    return launch_sample_polya_ps(d_rk, a, IPFE_N, 3, q, st);
}

int launch_sample_polya_ps(const uint32_t *d_rk, uint32_t *a, int n, int nmod, const uint32_t *q, hipStream_t st)
{
    if (n < 512 || (n & (n - 1)) || nmod < 1 || nmod > 4) {
        ipfe_set_error("sample_polya: unsupported shape n=%d nmod=%d", n, nmod);
        return -1;
    }
    PolyaArgs pa{};
    pa.n = n;
    pa.nmod = nmod;
    for (int s = 0; s < nmod; ++s) pa.q[s] = q[s];
    hipLaunchKernelGGL(k_sample_polya, dim3((unsigned)(n / 2 / 256)), dim3(256), 0, st, d_rk, g_aes_te, a, pa);
    HIP_OK(hipGetLastError());
    return 0;
}

int launch_aes_ctr(const uint32_t *d_rk, uint32_t nonce, uint32_t ctr0, uint32_t nblocks, uint8_t *out, hipStream_t st)
{
    if (nblocks == 0) return 0;
    hipLaunchKernelGGL(k_aes_ctr, dim3((nblocks + 255) / 256), dim3(256), 0, st, d_rk, g_aes_te, nonce, ctr0, nblocks,
                       (uint32_t *)out);
    HIP_OK(hipGetLastError());
    return 0;
}

}  // namespace ipfe
