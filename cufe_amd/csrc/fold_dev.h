// fold_dev.h -- the fold  acc <- mod_prime(y_i v_i + acc)  of key generation and
// decryption as a plain sum, for k_scheme.hip and k_pset.hip.
//
// mod_prime returns the canonical residue unless its argument is a multiple of
// the modulus, so the fold's result is the canonical sum (FoldSum) wherever that
// is not zero; where it is, 0 or q by the fold's last steps (fold_zero).
#pragma once
#include "ipfe_common.h"

namespace ipfe {

// sum of y v for y < 2^31; at most 65,536 terms
struct FoldSum {
    uint64_t lo = 0, hi = 0;
    __device__ __forceinline__ void add(uint32_t y, uint32_t v)
    {
        lo += (uint64_t)(y & 0xffffu) * v;
        if (y >> 16) hi += (uint64_t)(y >> 16) * v;
    }
    __device__ __forceinline__ uint32_t value(uint32_t q, uint32_t mu_hi, uint32_t mu_lo) const
    {
        const uint64_t h = hi ? reduce64(hi, q, mu_hi, mu_lo) : 0u;
        return reduce64(lo + (h << 16), q, mu_hi, mu_lo);
    }
};

// The fold's result where its sum is 0 mod q: entries 0 .. n-1 with term(e, y,
// v, i) giving y mod q, v and the slot i of entry e (ascending; slots between
// entries hold y = 0, which only map acc = q to 0), len slots; mod: mod_prime.
// Before the last entry whose product is not 0 mod q, acc is the canonical
// residue that cancels it, whatever came before; from there on the fold is run
// literally.  (Sums of small keys are 0 often enough, 10 coefficients of 128 keys
// over 785 slots, that running the whole fold there took that kernel 205 us
// instead of 62.)
template <class Mod, class Term>
__device__ uint32_t fold_zero(int n, int len, uint32_t q, Mod mod, Term term)
{
    uint32_t y, v;
    int i, e = n - 1;
    uint64_t t = 0;
    for (; e >= 0; --e) {
        term(e, y, v, i);
        t = (uint64_t)y * v % q;
        if (t) break;
    }
    uint32_t acc = e >= 0 ? q - (uint32_t)t : 0u;
    int last = -1;
    if (e >= 0) {
        acc = mod((uint64_t)y * v + acc);
        last = i;
    }
    for (++e; e < n; ++e) {
        term(e, y, v, i);
        if (i > last + 1 && acc == q) acc = 0;
        acc = mod((uint64_t)y * v + acc);
        last = i;
    }
    if (last < len - 1 && acc == q) acc = 0;
    return acc;
}

constexpr int FOLD_WAVES = 4;  // waves of a workgroup, each with its share of the terms

}  // namespace ipfe
