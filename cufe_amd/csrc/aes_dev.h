// aes_dev.h -- AES-256 encryption of CTR counter blocks with T-tables in LDS.
//
// Counter block of stream (key, nonce) at counter t is BE16(nonce) || 0^10 ||
// BE32(t) (the block layout src/aes256ctr.c:27-40 produces).  Round keys are
// the FIPS-197 big-endian words; the four T-tables (1 KiB each) are staged in
// LDS by the calling workgroup.  The output block is returned as four
// little-endian words, i.e. word w holds bytes 4w..4w+3 of the keystream, which
// is how every consumer reads it (LE32 / LE64 loads).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ipfe {

constexpr int AES_TABLE_WORDS = 4 * 256;

// a ^ b ^ c as one v_bitop3_b32 (truth table 0x96); the compiler does not
// form it from two XORs by itself.
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c)
{
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}

__device__ __forceinline__ void aes_stage_tables(uint32_t *lds_te, const uint32_t *__restrict__ te_global)
{
    for (int i = threadIdx.x; i < AES_TABLE_WORDS; i += blockDim.x) lds_te[i] = te_global[i];
}

// rk: 60 round-key words, uniform across the workgroup (scalar loads).
__device__ __forceinline__ void aes256_ctr_block(const uint32_t *__restrict__ rk, const uint32_t *te, uint32_t nonce,
                                                 uint32_t ctr, uint32_t (&o)[4])
{
    const uint32_t *T0 = te, *T1 = te + 256, *T2 = te + 512, *T3 = te + 768;
    uint32_t s0 = (nonce << 16) ^ rk[0];
    uint32_t s1 = rk[1];
    uint32_t s2 = rk[2];
    uint32_t s3 = ctr ^ rk[3];
#pragma unroll
    for (int r = 1; r < 14; ++r) {
        uint32_t t0 = xor3(xor3(T0[s0 >> 24], T1[(s1 >> 16) & 255], T2[(s2 >> 8) & 255]), T3[s3 & 255], rk[4 * r]);
        uint32_t t1 = xor3(xor3(T0[s1 >> 24], T1[(s2 >> 16) & 255], T2[(s3 >> 8) & 255]), T3[s0 & 255], rk[4 * r + 1]);
        uint32_t t2 = xor3(xor3(T0[s2 >> 24], T1[(s3 >> 16) & 255], T2[(s0 >> 8) & 255]), T3[s1 & 255], rk[4 * r + 2]);
        uint32_t t3 = xor3(xor3(T0[s3 >> 24], T1[(s0 >> 16) & 255], T2[(s1 >> 8) & 255]), T3[s2 & 255], rk[4 * r + 3]);
        s0 = t0; s1 = t1; s2 = t2; s3 = t3;
    }
    // Final round (SubBytes, ShiftRows, AddRoundKey): the S-box byte sits in
    // byte 3 of T2, byte 2 of T3, byte 1 of T0 and byte 0 of T1.
    uint32_t f0 = (T2[s0 >> 24] & 0xff000000u) ^ (T3[(s1 >> 16) & 255] & 0x00ff0000u) ^
                  (T0[(s2 >> 8) & 255] & 0x0000ff00u) ^ (T1[s3 & 255] & 0x000000ffu) ^ rk[56];
    uint32_t f1 = (T2[s1 >> 24] & 0xff000000u) ^ (T3[(s2 >> 16) & 255] & 0x00ff0000u) ^
                  (T0[(s3 >> 8) & 255] & 0x0000ff00u) ^ (T1[s0 & 255] & 0x000000ffu) ^ rk[57];
    uint32_t f2 = (T2[s2 >> 24] & 0xff000000u) ^ (T3[(s3 >> 16) & 255] & 0x00ff0000u) ^
                  (T0[(s0 >> 8) & 255] & 0x0000ff00u) ^ (T1[s1 & 255] & 0x000000ffu) ^ rk[58];
    uint32_t f3 = (T2[s3 >> 24] & 0xff000000u) ^ (T3[(s0 >> 16) & 255] & 0x00ff0000u) ^
                  (T0[(s1 >> 8) & 255] & 0x0000ff00u) ^ (T1[s2 & 255] & 0x000000ffu) ^ rk[59];
    o[0] = __builtin_bswap32(f0);
    o[1] = __builtin_bswap32(f1);
    o[2] = __builtin_bswap32(f2);
    o[3] = __builtin_bswap32(f3);
}

// Bank-replicated variant: T0 stored 32 times so that lane l reads copy
// l mod 32 -- entry x of copy c at word 32 x + c, i.e. in bank c, so the 32
// lanes of a half-wave never collide.  T1..T3 are rotations of T0.
constexpr int AES_REP_WORDS = 256 * 32;

__device__ __forceinline__ void aes_stage_tables_rep(uint32_t *lds_rep, const uint32_t *__restrict__ te_global)
{
    for (int i = threadIdx.x; i < AES_REP_WORDS; i += blockDim.x) lds_rep[i] = te_global[i >> 5];
}

__device__ __forceinline__ uint32_t ror32(uint32_t x, int n) { return __builtin_amdgcn_alignbit(x, x, n); }

__device__ __forceinline__ void aes256_ctr_block_rep(const uint32_t *__restrict__ rk, const uint32_t *te_rep,
                                                     uint32_t nonce, uint32_t ctr, uint32_t (&o)[4])
{
    const uint32_t *T = te_rep + (threadIdx.x & 31);
#define TL(x) T[(x) << 5]
    uint32_t s0 = (nonce << 16) ^ rk[0];
    uint32_t s1 = rk[1];
    uint32_t s2 = rk[2];
    uint32_t s3 = ctr ^ rk[3];
#pragma unroll
    for (int r = 1; r < 14; ++r) {
        uint32_t t0 = xor3(xor3(TL(s0 >> 24), ror32(TL((s1 >> 16) & 255), 8), ror32(TL((s2 >> 8) & 255), 16)),
                           ror32(TL(s3 & 255), 24), rk[4 * r]);
        uint32_t t1 = xor3(xor3(TL(s1 >> 24), ror32(TL((s2 >> 16) & 255), 8), ror32(TL((s3 >> 8) & 255), 16)),
                           ror32(TL(s0 & 255), 24), rk[4 * r + 1]);
        uint32_t t2 = xor3(xor3(TL(s2 >> 24), ror32(TL((s3 >> 16) & 255), 8), ror32(TL((s0 >> 8) & 255), 16)),
                           ror32(TL(s1 & 255), 24), rk[4 * r + 2]);
        uint32_t t3 = xor3(xor3(TL(s3 >> 24), ror32(TL((s0 >> 16) & 255), 8), ror32(TL((s1 >> 8) & 255), 16)),
                           ror32(TL(s2 & 255), 24), rk[4 * r + 3]);
        s0 = t0; s1 = t1; s2 = t2; s3 = t3;
    }
    // S-box byte of T0[x] is byte 1 (and byte 2)
    uint32_t f0 = ((TL(s0 >> 24) << 16) & 0xff000000u) ^ (TL((s1 >> 16) & 255) & 0x00ff0000u) ^
                  (TL((s2 >> 8) & 255) & 0x0000ff00u) ^ ((TL(s3 & 255) >> 8) & 0xffu) ^ rk[56];
    uint32_t f1 = ((TL(s1 >> 24) << 16) & 0xff000000u) ^ (TL((s2 >> 16) & 255) & 0x00ff0000u) ^
                  (TL((s3 >> 8) & 255) & 0x0000ff00u) ^ ((TL(s0 & 255) >> 8) & 0xffu) ^ rk[57];
    uint32_t f2 = ((TL(s2 >> 24) << 16) & 0xff000000u) ^ (TL((s3 >> 16) & 255) & 0x00ff0000u) ^
                  (TL((s0 >> 8) & 255) & 0x0000ff00u) ^ ((TL(s1 & 255) >> 8) & 0xffu) ^ rk[58];
    uint32_t f3 = ((TL(s3 >> 24) << 16) & 0xff000000u) ^ (TL((s0 >> 16) & 255) & 0x00ff0000u) ^
                  (TL((s1 >> 8) & 255) & 0x0000ff00u) ^ ((TL(s2 & 255) >> 8) & 0xffu) ^ rk[59];
#undef TL
    o[0] = __builtin_bswap32(f0);
    o[1] = __builtin_bswap32(f1);
    o[2] = __builtin_bswap32(f2);
    o[3] = __builtin_bswap32(f3);
}

// Table layouts for the generic round code below.  A round word
//   T0[a] ^ T1[b] ^ T2[c] ^ T3[d] ^ key,  T1..T3 = T0 rotated right by 8, 16, 24,
// is word(): from T0 and T2 alone it is
//   (T0[a] ^ T2[c]) ^ ror8(T0[b] ^ T2[d]) ^ key,
// one rotation when T2 is a table of its own, none with all four.  t0(w, k)
// and t2(w, k) look byte k of w up in T0 and T2; the S-box byte is byte 1 (and
// 2) of a T0 entry.
template <class Tab>
struct AesTwo {  // round word from t0 and t2
    __device__ uint32_t word(uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t key) const
    {
        const Tab &t = static_cast<const Tab &>(*this);
        return xor3(t.t0(a, 3), t.t2(c, 1), key) ^ ror32(t.t0(b, 2) ^ t.t2(d, 0), 8);
    }
};

struct AesTab4 {  // the four 1 KiB tables, no replication
    const uint32_t *T;
    __device__ explicit AesTab4(const uint32_t *te) : T(te) {}
    __device__ uint32_t t0(uint32_t w, int k) const { return T[(w >> (8 * k)) & 255]; }
    __device__ uint32_t t2(uint32_t w, int k) const { return T[512 + ((w >> (8 * k)) & 255)]; }
    __device__ uint32_t word(uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t key) const
    {
        return xor3(xor3(T[a >> 24], T[256 + ((b >> 16) & 255)], T[512 + ((c >> 8) & 255)]), T[768 + (d & 255)], key);
    }
};

struct AesTabRep : AesTwo<AesTabRep> {  // T0 only, bank-replicated (32 KiB): entry x of copy c at word 32 x + c
    const uint32_t *T;
    __device__ explicit AesTabRep(const uint32_t *te) : T(te + (threadIdx.x & 31)) {}
    __device__ uint32_t t0(uint32_t w, int k) const { return T[((w >> (8 * k)) & 255) << 5]; }
    __device__ uint32_t t2(uint32_t w, int k) const { return ror32(t0(w, k), 16); }
};

// T0 and T2, bank-replicated (64 KiB): entry x of copy c at word 64 x + c
// (T0) and 64 x + 32 + c (T2).  The byte address 256 x + 4 c (+ 128) is one
// v_perm_b32: byte 0 from the lane's offset, byte 1 = byte k of w.
constexpr int AES_REP2_WORDS = 256 * 64;
struct AesTabRep2 : AesTwo<AesTabRep2> {
    const char *base;
    uint32_t l0, l2;
    __device__ explicit AesTabRep2(const uint32_t *te)
        : base(reinterpret_cast<const char *>(te)), l0(4u * (threadIdx.x & 31)), l2(128u + 4u * (threadIdx.x & 31))
    {
    }
    __device__ uint32_t t0(uint32_t w, int k) const
    {
        return *reinterpret_cast<const uint32_t *>(base + __builtin_amdgcn_perm(w, l0, 0x0C0C0400u | ((4u + k) << 8)));
    }
    __device__ uint32_t t2(uint32_t w, int k) const
    {
        return *reinterpret_cast<const uint32_t *>(base + __builtin_amdgcn_perm(w, l2, 0x0C0C0400u | ((4u + k) << 8)));
    }
};

// All four tables, bank-replicated (128 KiB): T0 and T2 as above, T1 and T3
// likewise in the second 64 KiB (byte 2 of the lane's offset is 1): every
// lookup address is one v_perm_b32 and no word is rotated -- 24 VALU
// instructions a round against 32 with two tables, beside 16 lookups that
// take the LDS 32 cycles of a CU.
constexpr int AES_REP4_WORDS = 256 * 128;
struct AesTabRep4 {
    const char *base;
    uint32_t l0, l1, l2, l3;
    __device__ explicit AesTabRep4(const uint32_t *te) : base(reinterpret_cast<const char *>(te))
    {
        l0 = 4u * (threadIdx.x & 31);
        l2 = l0 + 128u;
        l1 = l0 + 65536u;
        l3 = l2 + 65536u;
    }
    __device__ uint32_t at(uint32_t w, int k, uint32_t l, uint32_t top) const
    {
        return *reinterpret_cast<const uint32_t *>(base + __builtin_amdgcn_perm(w, l, top | ((4u + k) << 8)));
    }
    __device__ uint32_t t0(uint32_t w, int k) const { return at(w, k, l0, 0x0C0C0000u); }
    __device__ uint32_t t2(uint32_t w, int k) const { return at(w, k, l2, 0x0C0C0000u); }
    __device__ uint32_t word(uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t key) const
    {
        return xor3(xor3(t0(a, 3), at(b, 2, l1, 0x0C020000u), t2(c, 1)), at(d, 0, l3, 0x0C020000u), key);
    }
};

__device__ __forceinline__ void aes_stage_tables_rep2(uint32_t *lds, const uint32_t *__restrict__ te_global)
{
    for (int i = threadIdx.x; i < AES_REP2_WORDS; i += blockDim.x) {
        const uint32_t v = te_global[i >> 6];
        lds[i] = (i & 32) ? ror32(v, 16) : v;
    }
}

__device__ __forceinline__ void aes_stage_tables_rep4(uint32_t *lds, const uint32_t *__restrict__ te_global)
{
    for (int i = threadIdx.x; i < AES_REP4_WORDS / 4; i += blockDim.x) {
        const int half = i >> 12, two = (i >> 3) & 1;  // 16 words of four copies per entry
        const uint32_t v = te_global[256 * (half + 2 * two) + ((i >> 4) & 255)];
        reinterpret_cast<uint4 *>(lds)[i] = make_uint4(v, v, v, v);
    }
}

// One middle round with round-key words rk[0..3].
template <class Tab, class Rk>
__device__ __forceinline__ void aes_round(const Tab &tb, uint32_t &s0, uint32_t &s1, uint32_t &s2, uint32_t &s3, Rk rk)
{
    const uint32_t t0 = tb.word(s0, s1, s2, s3, rk[0]);
    const uint32_t t1 = tb.word(s1, s2, s3, s0, rk[1]);
    const uint32_t t2 = tb.word(s2, s3, s0, s1, rk[2]);
    const uint32_t t3 = tb.word(s3, s0, s1, s2, rk[3]);
    s0 = t0;
    s1 = t1;
    s2 = t2;
    s3 = t3;
}

// An output word of the final round (SubBytes, ShiftRows, AddRoundKey) in the
// keystream's byte order: S[a's byte 3], S[b's 2], S[c's 1], S[d's 0] from the
// low byte up, each the byte 1 of a T0 entry; key: the byte-swapped key word.
template <class Tab>
__device__ __forceinline__ uint32_t aes_last(const Tab &tb, uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t key)
{
    const uint32_t lo = __builtin_amdgcn_perm(tb.t0(a, 3), tb.t0(b, 2), 0x0C0C0105u);
    const uint32_t hi = __builtin_amdgcn_perm(tb.t0(c, 1), tb.t0(d, 0), 0x01050C0Cu);
    return xor3(lo, hi, key);
}

// Rounds 3..14 from the state after round 2; rkf: the last four round-key
// words, byte-swapped.  WORDS: the output words to form (bit j: o[j]).
template <int WORDS = 15, class Tab, class Rk>
__device__ __forceinline__ void aes_rounds_from3(const Tab &tb, uint32_t s0, uint32_t s1, uint32_t s2, uint32_t s3,
                                                 Rk rk, Rk rkf, uint32_t (&o)[4])
{
#pragma unroll
    for (int r = 3; r < 14; ++r) aes_round(tb, s0, s1, s2, s3, rk + 4 * r);
    if (WORDS & 1) o[0] = aes_last(tb, s0, s1, s2, s3, rkf[0]);
    if (WORDS & 2) o[1] = aes_last(tb, s1, s2, s3, s0, rkf[1]);
    if (WORDS & 4) o[2] = aes_last(tb, s2, s3, s0, s1, rkf[2]);
    if (WORDS & 8) o[3] = aes_last(tb, s3, s0, s1, s2, rkf[3]);
}

// Block at counter ctr of stream (rk, nonce).
template <int WORDS = 15, class Tab, class Rk>
__device__ __forceinline__ void aes256_ctr_block_t(const Tab &tb, Rk rk, Rk rkf, uint32_t nonce, uint32_t ctr,
                                                   uint32_t (&o)[4])
{
    uint32_t s0 = (nonce << 16) ^ rk[0], s1 = rk[1], s2 = rk[2], s3 = ctr ^ rk[3];
    aes_round(tb, s0, s1, s2, s3, rk + 4);
    aes_round(tb, s0, s1, s2, s3, rk + 8);
    aes_rounds_from3<WORDS>(tb, s0, s1, s2, s3, rk, rkf, o);
}

// Counter-mode shortcut.  The counter sits in state word 3, so in round 1
// only the lookup of its low byte changes between the 256 counters that share
// bits 8..31: t0 = C0 ^ ror8(T2[(ctr ^ rk3) & 255]), and t1..t3 are constant.
// In round 2 each output word then has one lookup that depends on t0 and the
// rest do not.  aes256_ctr_window computes, once per such window of counters,
// w = {C0, t1, t2, t3, D0..D3} with D_j the constant part of round-2 word j;
// aes256_ctr_block_win finishes a block from it with 5 lookups in rounds 1-2
// instead of 32.  Both give the block of aes256_ctr_block_t.
template <class Tab, class Rk>
__device__ __forceinline__ void aes256_ctr_window(const Tab &tb, Rk rk, uint32_t nonce, uint32_t ctr_hi, uint32_t *w)
{
    const uint32_t s0 = (nonce << 16) ^ rk[0], s1 = rk[1], s2 = rk[2], s3 = (ctr_hi << 8) ^ rk[3];
    const uint32_t t1 = tb.t0(s1, 3) ^ tb.t2(s3, 1) ^ ror32(tb.t0(s2, 2) ^ tb.t2(s0, 0), 8) ^ rk[5];
    const uint32_t t2 = tb.t0(s2, 3) ^ tb.t2(s0, 1) ^ ror32(tb.t0(s3, 2) ^ tb.t2(s1, 0), 8) ^ rk[6];
    const uint32_t t3 = tb.t0(s3, 3) ^ tb.t2(s1, 1) ^ ror32(tb.t0(s0, 2) ^ tb.t2(s2, 0), 8) ^ rk[7];
    w[0] = tb.t0(s0, 3) ^ tb.t2(s2, 1) ^ ror32(tb.t0(s1, 2), 8) ^ rk[4];
    w[1] = t1;
    w[2] = t2;
    w[3] = t3;
    w[4] = tb.t2(t2, 1) ^ ror32(tb.t0(t1, 2) ^ tb.t2(t3, 0), 8) ^ rk[8];
    w[5] = tb.t0(t1, 3) ^ tb.t2(t3, 1) ^ ror32(tb.t0(t2, 2), 8) ^ rk[9];
    w[6] = tb.t0(t2, 3) ^ ror32(tb.t0(t3, 2) ^ tb.t2(t1, 0), 8) ^ rk[10];
    w[7] = tb.t0(t3, 3) ^ tb.t2(t1, 1) ^ ror32(tb.t2(t2, 0), 8) ^ rk[11];
}

template <int WORDS = 15, class Tab, class Rk>
__device__ __forceinline__ void aes256_ctr_block_win(const Tab &tb, Rk rk, Rk rkf, const uint32_t *w, uint32_t ctr,
                                                     uint32_t (&o)[4])
{
    const uint32_t t0 = w[0] ^ ror32(tb.t2(ctr ^ rk[3], 0), 8);
    const uint32_t s0 = tb.t0(t0, 3) ^ w[4];
    const uint32_t s1 = ror32(tb.t2(t0, 0), 8) ^ w[5];
    const uint32_t s2 = tb.t2(t0, 1) ^ w[6];
    const uint32_t s3 = ror32(tb.t0(t0, 2), 8) ^ w[7];
    aes_rounds_from3<WORDS>(tb, s0, s1, s2, s3, rk, rkf, o);
}

}  // namespace ipfe
