// kernels.h -- launch wrappers of the gfx950 kernels (host side, C++ linkage).
// Every launcher returns 0 or -1 with the error text set through ipfe_set_error.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>

#include "ipfe_common.h"

namespace ipfe {

struct NinvConsts {
    uint32_t ninv[3], ninvp[3], flag[3];
};
struct ScaleConsts {
    uint32_t scale[3];  // floor(Q/p) mod q_j
};
struct BarrettConsts {
    uint32_t mu_hi[3], mu_lo[3];
};

// ----- NTT domain (k_ntt.hip) -----
struct EncMsg {
    const uint32_t *x;      // message [len]
    const uint32_t *rhat;   // NTT(r) [3][N]
    const uint32_t *rhatp;  // Shoup companions of rhat
    uint32_t *c;            // c_0 .. c_{len-1} [len][3][N]; hold the noise f on entry
    uint32_t *cl;           // c_L [3][N]; holds f_0 on entry
    int len;
    int pad;
};
struct EncItem {
    int msg, poly;
};

int launch_ntt_fwd(const uint32_t *in, uint32_t *out, int npoly_limbs, const uint32_t *tw_all, hipStream_t st);
int launch_ntt_inv(const uint32_t *in, uint32_t *out, int npoly_limbs, const uint32_t *tw_all, const NinvConsts &nc,
                   hipStream_t st);
int launch_shoup_prep(const uint32_t *v, uint32_t *vp, size_t n_total, hipStream_t st);
int launch_setup_pk(const uint32_t *msk, const uint32_t *e, const uint32_t *ahat, const uint32_t *ahatp, uint32_t *mpk,
                    int l, const uint32_t *tw_all, hipStream_t st);
int launch_enc_poly(const EncItem *items, int nitems, const EncMsg *msgs, const uint32_t *mpk, int mpk_l,
                    const uint32_t *tw_all, const NinvConsts &nc, const ScaleConsts &sc, hipStream_t st);
// d[v] = sub_mod(d[v], poly_mul_ntt(c_L, sk[v])) for nvec keys; chat = NTT(c_L)
// [3][N], sk and d [nvec][3][N].
int launch_dec_poly(const uint32_t *chat, const uint32_t *sk, uint32_t *d, int nvec, const uint32_t *tw_all,
                    const NinvConsts &nc, const BarrettConsts &bc, hipStream_t st);

// ----- Sampler (k_sampler.hip) -----
// One AES-256-CTR Gaussian stream cut into 384-byte chunks (24 AES blocks).
// Chunk c of the stream uses counters 24c .. 24c+23.  Calls take slen accepted
// candidates each; call 0 writes to out0, call k >= 1 to out1 + (k-1)*out_stride.
struct GaussStream {
    uint32_t rk[60];         // expanded AES-256 key
    uint32_t rkf[4];         // its last four words, byte-swapped
    uint32_t nonce;          // 16-bit nonce
    int which;               // sampler width index into the device tables: 1, 2, 3 (S1, S2, S3 of the
                             // reference set), 4, 5 (the S2 / S3 widths of the N = 2048 set)
    int ncalls;              // number of calls
    int nchunks;             // speculative window length (chunks)
    long long chunk_base;    // index of this stream's chunk 0 in the chunk arrays
    uint32_t *out0;          // [nmod][slen] destination of call 0
    uint32_t *out1;          // destination of call 1
    long long out_stride;    // words between consecutive calls from call 1 on
    int coef0_only;          // 1: write only sample 0 of each call, nmod words at out0 + nmod*call
    int slen;                // samples per call (the parameter set's N)
    long long first_base;    // compact streams: index of call 0 in the per-call first-chunk array
    uint32_t q[4];           // output moduli, limbs 0 .. nmod-1
    uint32_t fold[4];        // mod_prime fold shifts per limb: a | b << 8 (q = 2^a - 2^b + 1)
    int nmod;                // output limbs
    int span;                // chunks a call may span (a longer one counts as a short window)
    long long map_base;      // compact streams: first word of the stream's maps in the walk's map array
};

// Candidate pass: for every chunk of every stream, AES + CDT + Bernoulli;
// writes the accepted count and the accepted (z | sign << 63) values in order.
// chunk_prefix: each stream's first chunk, multiples of 16, as is nchunks_total.
// full: a chunk whose uniform scan runs past the words the default AES blocks
// hold is scanned on (else it sets status bit 4)
int launch_gauss_candidates(const GaussStream *d_streams, int nstreams, const long long *d_chunk_prefix,
                            long long nchunks_total, uint8_t *cnt, uint64_t *vals, int *status, int full,
                            hipStream_t st);
// Walk (k_gauss_walk.hip): per stream, the call boundaries from the counts;
// writes per chunk of the full streams (call << 13 | offset) or -1, padding
// included.  status[stream] = 1 when the window was short (else it stays).
// Streams start on a multiple of 16 chunks and pad their last to one; map
// holds span words per window of GAUSS_WALK_WIN chunks of the compact
// streams (full streams keep theirs in pos); max_chunks: the longest window.
constexpr int GAUSS_WALK_WIN = 16384;
int launch_gauss_walk(const GaussStream *d_streams, int nstreams, int max_chunks, const uint8_t *cnt, int *pos,
                      uint32_t *map, long long *firsts, int *status, hipStream_t st);
// Compact streams: recompute the first non-empty chunk of every call and write sample 0.
int launch_gauss_firsts(const GaussStream *d_streams, int nstreams, const long long *d_first_prefix,
                        const long long *firsts, long long nitems, int *status, int full, hipStream_t st);
int launch_gauss_scatter(const GaussStream *d_streams, int nstreams, const long long *d_chunk_prefix,
                         long long nchunks_total, const uint8_t *cnt, const uint64_t *vals, const int *pos,
                         hipStream_t st);
int launch_fill_i32(int *p, int v, size_t n, hipStream_t st);

// Uniform polynomial a (src/sample.c:56-128) on device from the expanded key.
int launch_sample_polya(const uint32_t *d_rk, uint32_t *a, hipStream_t st);
// The same for any parameter set: n coefficients on nmod limbs of moduli q.
int launch_sample_polya_ps(const uint32_t *d_rk, uint32_t *a, int n, int nmod, const uint32_t *q, hipStream_t st);
// Raw keystream (tests): nblocks AES blocks from counter ctr0.
int launch_aes_ctr(const uint32_t *d_rk, uint32_t nonce, uint32_t ctr0, uint32_t nblocks, uint8_t *out, hipStream_t st);

// ----- Keys, decryption, CRT (k_scheme.hip) -----
// Sparse description of vectors y: for vector v, entries [off[v], off[v+1]) of
// (idx, val) with idx ascending; len = the slot count the reference loops over.
struct SparseY {
    const int *off;
    const int *idx;
    const uint32_t *val;
    int len;
    // the vectors themselves [nvec][len] where fold_dense holds, and scratch of
    // fold_packed_words(nvec, len)
    const uint32_t *dense = nullptr;
    uint32_t *dense_packed = nullptr;
};
// The lists of dense vectors y [n][stride] (device): off [n + 1] and info first
// (info[0]: the largest slot in use plus one, info[1]: v stride + i of the first
// entry at a slot i >= limit, or ~0, info[2]: the entries), then idx and val.
int launch_sparse_count(const uint32_t *y, int n, int stride, int limit, int *off, unsigned int *info, hipStream_t st);
int launch_sparse_fill(const uint32_t *y, int n, int stride, const int *off, int *idx, uint32_t *val, hipStream_t st);
// out[v][3][N] = sum_i y_v[i] P[i] with the reference's sequential fold: keygen
// (P = msk) and the first half of rlwe_sife_decrypt_gmp (P = c).
int launch_fold(const SparseY &y, int nvec, const uint32_t *P, uint32_t *out, const BarrettConsts &bc,
                hipStream_t st);
// Whether vectors with nnz entries in all, none above max_y, take the dense form.
bool fold_dense(size_t nvec, size_t len, size_t nnz, uint32_t max_y);
size_t fold_packed_words(size_t nvec, size_t len);
// CRT + rounding of coefficient k of d[v][3][N] -> r[v]  (k = 0 for kvalues).
int launch_crt_round(const uint32_t *d, int nvec, int coef, uint32_t *r, hipStream_t st);
// out += sum over i of (2i+1) * w[i] mod 2^64 (out must be cleared first)
int launch_checksum(const uint32_t *w, size_t n, unsigned long long *out, hipStream_t st);

}  // namespace ipfe
