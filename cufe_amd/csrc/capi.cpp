// capi.cpp -- the C ABI of include/cufe_ipfe.h: reference drop-ins, host helpers
// and single-operation entry points.
#include <stdio.h>
#include <string.h>

#include <cmath>
#include <vector>

#include "../../include/cufe_ipfe.h"
#include "crt_dev.h"
#include "runtime.h"
#include "kernels_pset.h"

using namespace ipfe;

namespace {

constexpr size_t kPoly = (size_t)3 * IPFE_N;  // words per [3][N] polynomial

struct EventTimer {
    hipEvent_t a = nullptr, b = nullptr;
    hipStream_t st;
    explicit EventTimer(hipStream_t s, bool on = true) : st(s)
    {
        if (!on) return;
        (void)hipEventCreate(&a);
        (void)hipEventCreate(&b);
        (void)hipEventRecord(a, st);
    }
    float stop()
    {
        float ms = 0;
        if (!a) return ms;
        (void)hipEventRecord(b, st);
        (void)hipEventSynchronize(b);
        (void)hipEventElapsedTime(&ms, a, b);
        return ms;
    }
    ~EventTimer()
    {
        if (a) (void)hipEventDestroy(a);
        if (b) (void)hipEventDestroy(b);
    }
};

void report(const char *fn)
{
    fprintf(stderr, "[cufe_ipfe] %s failed: %s\n", fn, cufe_last_error());
}

// Sparse form of dense vectors y[n][len] (entries with y != 0, ascending).
struct HostSparse {
    std::vector<int> off, idx;
    std::vector<uint32_t> val;
    bool dense = false;
};
HostSparse to_sparse(const uint32_t *y, int n, int len)
{
    HostSparse h;
    h.off.resize(n + 1);
    for (int v = 0; v < n; ++v) {
        h.off[v] = (int)h.idx.size();
        for (int i = 0; i < len; ++i)
            if (y[(size_t)v * len + i]) {
                h.idx.push_back(i);
                h.val.push_back(y[(size_t)v * len + i]);
            }
    }
    h.off[n] = (int)h.idx.size();
    uint32_t max_y = 0;
    for (uint32_t v : h.val) max_y = std::max(max_y, v);
    h.dense = fold_dense((size_t)n, (size_t)len, h.idx.size(), max_y);
    if (h.idx.empty()) {  // keep device pointers valid
        h.idx.push_back(0);
        h.val.push_back(0);
    }
    return h;
}

struct DevSparse {
    DevBuf<int> off, idx;
    DevBuf<uint32_t> val;
    SparseY view{};
    // y [n][len]: the vectors h was made from
    int upload(const HostSparse &h, const uint32_t *y, int n, int len, hipStream_t st)
    {
        view.len = len;
        if (h.dense) {
            if (val.alloc((size_t)n * len + fold_packed_words(n, len))) return -1;
            if (copy_to_device(val.get(), y, (size_t)n * len * 4, st)) return -1;
            view.dense = val.get();
            view.dense_packed = val.get() + (size_t)n * len;
            return 0;
        }
        if (off.alloc(h.off.size()) || idx.alloc(h.idx.size()) || val.alloc(h.val.size())) return -1;
        HIP_OK(hipMemcpyAsync(off.get(), h.off.data(), h.off.size() * 4, hipMemcpyHostToDevice, st));
        HIP_OK(hipMemcpyAsync(idx.get(), h.idx.data(), h.idx.size() * 4, hipMemcpyHostToDevice, st));
        HIP_OK(hipMemcpyAsync(val.get(), h.val.data(), h.val.size() * 4, hipMemcpyHostToDevice, st));
        view.off = off.get();
        view.idx = idx.get();
        view.val = val.get();
        return 0;
    }
};

// ---------------------------------------------------------------------------
int do_setup(uint32_t *mpk, uint32_t *msk, const unsigned char *seed2, const unsigned char *seed3, int l, float *ms)
{
    Device *dev = device();
    if (!dev) return -1;
    hipStream_t st = dev->stream;
    EventTimer tm(st, ms != nullptr);
    DevBuf<uint32_t> d_mpk, d_msk, d_e, d_ap;
    if (d_mpk.alloc((l + 1) * kPoly) || d_msk.alloc(l * kPoly) || d_e.alloc(l * kPoly) || d_ap.alloc(kPoly)) return -1;
    uint32_t *d_ahat = d_mpk.get() + (size_t)l * kPoly;
    if (copy_to_device(d_ahat, mpk + (size_t)l * kPoly, kPoly * 4, st)) return -1;
    if (launch_ntt_fwd(d_ahat, d_ahat, 3, dev->tw_all, st)) return -1;
    if (launch_shoup_prep(d_ahat, d_ap.get(), kPoly, st)) return -1;
    std::vector<StreamReq> reqs;
    reqs.push_back(make_stream(seed2, 0, 1, l, d_msk.get(), d_msk.get() + kPoly, (long long)kPoly));
    reqs.push_back(make_stream(seed3, 0, 1, l, d_e.get(), d_e.get() + kPoly, (long long)kPoly));
    if (run_gauss(reqs, st)) return -1;
    if (launch_setup_pk(d_msk.get(), d_e.get(), d_ahat, d_ap.get(), d_mpk.get(), l, dev->tw_all, st)) return -1;
    if (copy_to_host(mpk, d_mpk.get(), (l + 1) * kPoly * 4, st)) return -1;
    if (copy_to_host(msk, d_msk.get(), l * kPoly * 4, st)) return -1;
    float e = tm.stop();
    if (ms) *ms += e;
    return sync_stream(st);
}

// Encrypt `repeat` messages of length l against mpk [l+1][3][N]; c is
// [repeat][l+1][3][N].  Message b uses nonce nonce0 + b.
int do_encrypt(const uint32_t *m, const uint32_t *mpk, uint32_t *c, const unsigned char *seed2,
               const unsigned char *seed3, int repeat, int l, int nonce0, float *ms)
{
    Device *dev = device();
    if (!dev) return -1;
    if (repeat < 0 || nonce0 < 0 || nonce0 + repeat > 65536) {
        ipfe_set_error("encrypt: nonce range [%d, %d) exceeds the 16-bit nonce space", nonce0, nonce0 + repeat);
        return -1;
    }
    hipStream_t st = dev->stream;
    EventTimer tm(st, ms != nullptr);
    DevBuf<uint32_t> d_mpk;
    if (d_mpk.alloc((l + 1) * kPoly)) return -1;
    // 39 MB at 785 slots, of use to launch_enc_poly only: uploaded beside the
    // sampling, which takes 0.4 ms: the whole call 2.47 ms, 2.81 with one after the other
    auto upload_mpk = [&] { return copy_to_device_beside(d_mpk.get(), mpk, (l + 1) * kPoly * 4, st); };
    const size_t ct_words = (size_t)(l + 1) * kPoly;
    // messages per group: bound ciphertext + sampler scratch to ~16 GiB
    const size_t per_msg = ct_words * 4 + gauss_bytes(3, l, 0) + gauss_bytes(2, 2, 0) + 2 * kPoly * 4;
    int group = (int)std::max<size_t>(1, ((size_t)16 << 30) / per_msg);
    for (int b0 = 0; b0 < repeat; b0 += group) {
        const int g = std::min(group, repeat - b0);
        DevBuf<uint32_t> d_x, d_c, d_r, d_rp;
        DevBuf<EncMsg> d_msgs;
        DevBuf<EncItem> d_items;
        if (d_x.alloc((size_t)g * l + 1) || d_c.alloc((size_t)g * ct_words) || d_r.alloc((size_t)g * kPoly) ||
            d_rp.alloc((size_t)g * kPoly) || d_msgs.alloc(g) || d_items.alloc((size_t)g * (l + 1)))
            return -1;
        if (l > 0)
            if (copy_to_device(d_x.get(), m + (size_t)b0 * l, (size_t)g * l * 4, st)) return -1;
        std::vector<StreamReq> reqs;
        std::vector<EncMsg> msgs(g);
        std::vector<EncItem> items;
        for (int b = 0; b < g; ++b) {
            uint32_t *cb = d_c.get() + (size_t)b * ct_words;
            const uint16_t nonce = (uint16_t)(nonce0 + b0 + b);
            // r, f_0 on (seed2, nonce); f_0 lands in the c_L slot
            reqs.push_back(make_stream(seed2, nonce, 2, 2, d_r.get() + (size_t)b * kPoly, cb + (size_t)l * kPoly, 0));
            if (l > 0) reqs.push_back(make_stream(seed3, nonce, 3, l, cb, cb + kPoly, (long long)kPoly));
            msgs[b].x = d_x.get() + (size_t)b * l;
            msgs[b].rhat = d_r.get() + (size_t)b * kPoly;
            msgs[b].rhatp = d_rp.get() + (size_t)b * kPoly;
            msgs[b].c = cb;
            msgs[b].cl = cb + (size_t)l * kPoly;
            msgs[b].len = l;
            for (int i = 0; i <= l; ++i) items.push_back(EncItem{b, i});
        }
        if (run_gauss(reqs, st, kGaussScratch, b0 ? std::function<int()>() : upload_mpk)) return -1;
        if (launch_ntt_fwd(d_r.get(), d_r.get(), g * 3, dev->tw_all, st)) return -1;
        if (launch_shoup_prep(d_r.get(), d_rp.get(), (size_t)g * kPoly, st)) return -1;
        HIP_OK(hipMemcpyAsync(d_msgs.get(), msgs.data(), sizeof(EncMsg) * g, hipMemcpyHostToDevice, st));
        HIP_OK(hipMemcpyAsync(d_items.get(), items.data(), sizeof(EncItem) * items.size(), hipMemcpyHostToDevice, st));
        if (launch_enc_poly(d_items.get(), (int)items.size(), d_msgs.get(), d_mpk.get(), l, dev->tw_all, dev->ninv,
                            dev->scale, st))
            return -1;
        if (copy_to_host(c + (size_t)b0 * ct_words, d_c.get(), (size_t)g * ct_words * 4, st)) return -1;
        if (sync_stream(st)) return -1;
    }
    float e = tm.stop();
    if (ms) *ms += e;
    return 0;
}

int do_keygen(const uint32_t *y, const uint32_t *msk, uint32_t *sk, int repeat, int l, float *ms)
{
    Device *dev = device();
    if (!dev) return -1;
    hipStream_t st = dev->stream;
    EventTimer tm(st, ms != nullptr);
    HostSparse hsp = to_sparse(y, repeat, l);
    DevSparse dsp;
    DevBuf<uint32_t> d_msk, d_sk;
    if (dsp.upload(hsp, y, repeat, l, st) || d_msk.alloc((size_t)l * kPoly + 1) || d_sk.alloc((size_t)repeat * kPoly)) return -1;
    if (l > 0 && copy_to_device(d_msk.get(), msk, (size_t)l * kPoly * 4, st)) return -1;
    if (launch_fold(dsp.view, repeat, d_msk.get(), d_sk.get(), dev->barrett, st)) return -1;
    if (copy_to_host(sk, d_sk.get(), (size_t)repeat * kPoly * 4, st)) return -1;
    float e = tm.stop();
    if (ms) *ms += e;
    return sync_stream(st);
}

// Decryption of c [l+1][3][N] under `repeat` keys, on the device: d [repeat][3][N].
// c's last polynomial is transformed in place.
int decrypt_dev(const SparseY &y, uint32_t *c, const uint32_t *sk, uint32_t *d, int repeat, int l, Device *dev,
                hipStream_t st)
{
    uint32_t *cl = c + (size_t)l * kPoly;
    if (launch_fold(y, repeat, c, d, dev->barrett, st)) return -1;
    // poly_mul_ntt(c_L, sk) (src/ntt.c:10-26): NTT both, pointwise, INTT
    if (launch_ntt_fwd(cl, cl, 3, dev->tw_all, st)) return -1;
    return launch_dec_poly(cl, sk, d, repeat, dev->tw_all, dev->ninv, dev->barrett, st);
}

// One ciphertext c [l+1][3][N] against `repeat` keys -> d_y [repeat][3][N].
int do_decrypt(const uint32_t *c, const uint32_t *y, const uint32_t *sk, uint32_t *d, int repeat, int l, float *ms)
{
    Device *dev = device();
    if (!dev) return -1;
    hipStream_t st = dev->stream;
    EventTimer tm(st, ms != nullptr);
    HostSparse hsp = to_sparse(y, repeat, l);
    DevSparse dsp;
    DevBuf<uint32_t> d_c, d_sk, d_d;
    if (dsp.upload(hsp, y, repeat, l, st) || d_c.alloc((size_t)(l + 1) * kPoly) || d_sk.alloc((size_t)repeat * kPoly) ||
        d_d.alloc((size_t)repeat * kPoly))
        return -1;
    if (copy_to_device(d_c.get(), c, (size_t)(l + 1) * kPoly * 4, st)) return -1;
    if (copy_to_device(d_sk.get(), sk, (size_t)repeat * kPoly * 4, st)) return -1;
    if (decrypt_dev(dsp.view, d_c.get(), d_sk.get(), d_d.get(), repeat, l, dev, st)) return -1;
    if (copy_to_host(d, d_d.get(), (size_t)repeat * kPoly * 4, st)) return -1;
    float e = tm.stop();
    if (ms) *ms += e;
    return sync_stream(st);
}

// Key values of one ciphertext c [L+1][3][N] under the keys of `n` vectors y
// [n][L]: key generation, decryption and the rounding of coefficient 0, with
// the keys and the decryptions kept on the device.
int do_kvalues(const uint32_t *c, const uint32_t *y, const uint32_t *msk, uint32_t *kv, int n)
{
    Device *dev = device();
    if (!dev) return -1;
    hipStream_t st = dev->stream;
    HostSparse hsp = to_sparse(y, n, IPFE_L);
    DevSparse dsp;
    DevBuf<uint32_t> d_msk, d_c, d_sk, d_d, d_kv;
    if (dsp.upload(hsp, y, n, IPFE_L, st) || d_msk.alloc(IPFE_L * kPoly) || d_c.alloc((IPFE_L + 1) * kPoly) ||
        d_sk.alloc((size_t)n * kPoly) || d_d.alloc((size_t)n * kPoly) || d_kv.alloc(n))
        return -1;
    if (copy_to_device(d_msk.get(), msk, IPFE_L * kPoly * 4, st)) return -1;
    if (launch_fold(dsp.view, n, d_msk.get(), d_sk.get(), dev->barrett, st)) return -1;
    if (copy_to_device(d_c.get(), c, (IPFE_L + 1) * kPoly * 4, st)) return -1;
    if (decrypt_dev(dsp.view, d_c.get(), d_sk.get(), d_d.get(), n, IPFE_L, dev, st)) return -1;
    if (launch_crt_round(d_d.get(), n, 0, d_kv.get(), st)) return -1;
    HIP_OK(hipMemcpyAsync(kv, d_kv.get(), (size_t)n * 4, hipMemcpyDeviceToHost, st));
    return sync_stream(st);
}

}  // namespace

// ===========================================================================
// 1. Reference drop-ins
// ===========================================================================
extern "C" void rlwe_sife_setup_gpu(uint32_t mpk[CUFE_SIFE_L + 1][CUFE_SIFE_NMODULI][CUFE_SIFE_N],
                                    uint32_t msk[CUFE_SIFE_L][CUFE_SIFE_NMODULI][CUFE_SIFE_N], unsigned char *seed2,
                                    unsigned char *seed3, float *part2_time)
{
    if (do_setup(&mpk[0][0][0], &msk[0][0][0], seed2, seed3, IPFE_L, part2_time)) report("rlwe_sife_setup_gpu");
}

extern "C" void rlwe_sife_encrypt_gpu(uint32_t *m, uint32_t mpk[CUFE_SIFE_L + 1][CUFE_SIFE_NMODULI][CUFE_SIFE_N],
                                      uint32_t *c, unsigned char *seed2, unsigned char *seed3, int repeat,
                                      float *part2_time)
{
    if (do_encrypt(m, &mpk[0][0][0], c, seed2, seed3, repeat, IPFE_L, 0, part2_time)) report("rlwe_sife_encrypt_gpu");
}

extern "C" void rlwe_sife_keygen_gpu(const uint32_t *y, const uint32_t msk[CUFE_SIFE_L][CUFE_SIFE_NMODULI][CUFE_SIFE_N],
                                     uint32_t *sk_y, int repeat, float *part2_time)
{
    if (do_keygen(y, &msk[0][0][0], sk_y, repeat, IPFE_L, part2_time)) report("rlwe_sife_keygen_gpu");
}

extern "C" void rlwe_sife_decrypt_gmp_gpu(uint32_t c[CUFE_SIFE_L + 1][CUFE_SIFE_NMODULI][CUFE_SIFE_N], const uint32_t *y,
                                          uint32_t *sk_y, uint32_t *d_y, int repeat, float *part2_time)
{
    if (do_decrypt(&c[0][0][0], y, sk_y, d_y, repeat, IPFE_L, part2_time)) report("rlwe_sife_decrypt_gmp_gpu");
}

// ===========================================================================
// 2. Host helpers
// ===========================================================================
extern "C" int cufe_sample_polya(const unsigned char seed[32], uint32_t *a)
{
    Device *dev = device();
    if (!dev) return -1;
    hipStream_t st = dev->stream;
    uint32_t rk[60];
    aes256_expand_key(seed, rk);
    DevBuf<uint32_t> d_rk, d_a;
    if (d_rk.alloc(60) || d_a.alloc(kPoly)) return -1;
    HIP_OK(hipMemcpyAsync(d_rk.get(), rk, sizeof rk, hipMemcpyHostToDevice, st));
    if (launch_sample_polya(d_rk.get(), d_a.get(), st)) return -1;
    if (copy_to_host(a, d_a.get(), kPoly * 4, st)) return -1;
    return sync_stream(st);
}

extern "C" double cufe_round_extract2(const uint32_t *d_y)
{
    return (double)crt_decode(d_y[0], d_y[IPFE_N], d_y[2 * IPFE_N]);
}

// svm_predict_gpu (main.c:270-390), plain per-call form.
extern "C" double cufe_svm_predict_gpu(const cufe_svm_model *model,
                                       uint32_t c[CUFE_SIFE_L + 1][CUFE_SIFE_NMODULI][CUFE_SIFE_N],
                                       const uint32_t msk[CUFE_SIFE_L][CUFE_SIFE_NMODULI][CUFE_SIFE_N], double *kvalue)
{
    if (!model || !c || !msk || model->l < 1 || model->nr_class < 2) {
        ipfe_set_error("cufe_svm_predict_gpu: bad arguments");
        return std::nan("");
    }
    const int l = model->l;
    // the steps of rlwe_sife_keygen_gpu and rlwe_sife_decrypt_gmp_gpu and the
    // rounding of the one coefficient that round_extract_gmp2 keeps, with their
    // status checked: a failed device call yields NaN, never a label voted from
    // unwritten key values
    std::vector<uint32_t> rounded(l);
    if (do_kvalues(&c[0][0][0], model->sv, &msk[0][0][0], rounded.data(), l)) {
        report("cufe_svm_predict_gpu");
        if (kvalue)
            for (int i = 0; i < l; ++i) kvalue[i] = std::nan("");
        return std::nan("");
    }
    std::vector<double> kv(rounded.begin(), rounded.end());
    if (kvalue) memcpy(kvalue, kv.data(), sizeof(double) * l);
    // one-vs-one vote (main.c:338-389)
    const int nr = model->nr_class;
    std::vector<int> start(nr), vote(nr, 0);
    start[0] = 0;
    for (int i = 1; i < nr; ++i) start[i] = start[i - 1] + model->nSV[i - 1];
    int p = 0;
    for (int i = 0; i < nr; ++i)
        for (int j = i + 1; j < nr; ++j) {
            double sum = 0;
            const double *coef1 = model->sv_coef + (size_t)(j - 1) * l;
            const double *coef2 = model->sv_coef + (size_t)i * l;
            for (int k = 0; k < model->nSV[i]; ++k) sum += coef1[start[i] + k] * kv[start[i] + k];
            for (int k = 0; k < model->nSV[j]; ++k) sum += coef2[start[j] + k] * kv[start[j] + k];
            sum -= model->rho[p];
            if (sum > 0) ++vote[i]; else ++vote[j];
            ++p;
        }
    int best = 0;
    for (int i = 1; i < nr; ++i)
        if (vote[i] > vote[best]) best = i;
    return model->label[best];
}

// ===========================================================================
// 3. Status-returning single operations
// ===========================================================================
extern "C" int cufe_device_info(char *name, int name_len, int *cu_count, uint64_t *hbm_bytes)
{
    hipDeviceProp_t prop;
    int d = 0;
    HIP_OK(hipGetDevice(&d));
    HIP_OK(hipGetDeviceProperties(&prop, d));
    if (name && name_len > 0) snprintf(name, (size_t)name_len, "%s (%s)", prop.name, prop.gcnArchName);
    if (cu_count) *cu_count = prop.multiProcessorCount;
    if (hbm_bytes) *hbm_bytes = prop.totalGlobalMem;
    return 0;
}

extern "C" int cufe_ntt_forward(uint32_t *polys, int npoly)
{
    Device *dev = device();
    if (!dev) return -1;
    hipStream_t st = dev->stream;
    DevBuf<uint32_t> d;
    if (d.alloc((size_t)npoly * kPoly)) return -1;
    if (copy_to_device(d.get(), polys, (size_t)npoly * kPoly * 4, st)) return -1;
    const PsetState *ps = pset_state(1);  // the reference set, tuned transform shape
    if (!ps || ps_ntt(*ps, false, d.get(), d.get(), npoly * 3, st)) return -1;
    if (copy_to_host(polys, d.get(), (size_t)npoly * kPoly * 4, st)) return -1;
    return sync_stream(st);
}

extern "C" int cufe_ntt_inverse(uint32_t *polys, int npoly)
{
    Device *dev = device();
    if (!dev) return -1;
    hipStream_t st = dev->stream;
    DevBuf<uint32_t> d;
    if (d.alloc((size_t)npoly * kPoly)) return -1;
    if (copy_to_device(d.get(), polys, (size_t)npoly * kPoly * 4, st)) return -1;
    const PsetState *ps = pset_state(1);
    if (!ps || ps_ntt(*ps, true, d.get(), d.get(), npoly * 3, st)) return -1;
    if (copy_to_host(polys, d.get(), (size_t)npoly * kPoly * 4, st)) return -1;
    return sync_stream(st);
}

extern "C" int cufe_gauss_sample(const unsigned char *keys, const uint16_t *nonces, int nstreams, int which, int ncalls,
                                 uint32_t *out)
{
    Device *dev = device();
    if (!dev) return -1;
    if (which < 1 || which > 3 || ncalls < 0 || nstreams < 0) {
        ipfe_set_error("cufe_gauss_sample: bad arguments (which=%d ncalls=%d nstreams=%d)", which, ncalls, nstreams);
        return -1;
    }
    if (ncalls == 0 || nstreams == 0) return 0;
    hipStream_t st = dev->stream;
    DevBuf<uint32_t> d;
    const size_t per_stream = (size_t)ncalls * kPoly;
    if (d.alloc((size_t)nstreams * per_stream)) return -1;
    std::vector<StreamReq> reqs;
    for (int t = 0; t < nstreams; ++t) {
        uint32_t *o = d.get() + (size_t)t * per_stream;
        reqs.push_back(make_stream(keys + 32 * (size_t)t, nonces[t], which, ncalls, o, o + kPoly, (long long)kPoly));
    }
    if (run_gauss(reqs, st)) return -1;
    if (copy_to_host(out, d.get(), (size_t)nstreams * per_stream * 4, st)) return -1;
    return sync_stream(st);
}

extern "C" int cufe_gauss_sample_first(const unsigned char *keys, const uint16_t *nonces, int nstreams, int which,
                                       int ncalls, uint32_t *out)
{
    Device *dev = device();
    if (!dev) return -1;
    if (which < 1 || which > 3 || ncalls < 0 || nstreams < 0) {
        ipfe_set_error("cufe_gauss_sample_first: bad arguments (which=%d ncalls=%d nstreams=%d)", which, ncalls,
                       nstreams);
        return -1;
    }
    if (ncalls == 0 || nstreams == 0) return 0;
    hipStream_t st = dev->stream;
    DevBuf<uint32_t> d;
    const size_t per_stream = (size_t)ncalls * 3;
    if (d.alloc((size_t)nstreams * per_stream)) return -1;
    std::vector<StreamReq> reqs;
    for (int t = 0; t < nstreams; ++t)
        reqs.push_back(make_stream(keys + 32 * (size_t)t, nonces[t], which, ncalls, d.get() + (size_t)t * per_stream,
                                   nullptr, 0, 1));
    if (run_gauss(reqs, st)) return -1;
    if (copy_to_host(out, d.get(), (size_t)nstreams * per_stream * 4, st)) return -1;
    return sync_stream(st);
}

extern "C" int cufe_aes256ctr(const unsigned char key[32], uint16_t nonce, uint32_t ctr0, uint32_t nblocks,
                              unsigned char *out)
{
    Device *dev = device();
    if (!dev) return -1;
    hipStream_t st = dev->stream;
    uint32_t rk[60];
    aes256_expand_key(key, rk);
    DevBuf<uint32_t> d_rk;
    DevBuf<uint8_t> d_out;
    if (d_rk.alloc(60) || d_out.alloc((size_t)nblocks * 16 + 16)) return -1;
    HIP_OK(hipMemcpyAsync(d_rk.get(), rk, sizeof rk, hipMemcpyHostToDevice, st));
    if (launch_aes_ctr(d_rk.get(), nonce, ctr0, nblocks, d_out.get(), st)) return -1;
    HIP_OK(hipMemcpyAsync(out, d_out.get(), (size_t)nblocks * 16, hipMemcpyDeviceToHost, st));
    return sync_stream(st);
}

extern "C" int cufe_crt_round(const uint32_t *d, int nvec, int coef, uint32_t *r)
{
    Device *dev = device();
    if (!dev) return -1;
    if (coef < 0 || coef >= IPFE_N) {
        ipfe_set_error("cufe_crt_round: coefficient %d out of range", coef);
        return -1;
    }
    hipStream_t st = dev->stream;
    DevBuf<uint32_t> d_d, d_r;
    if (d_d.alloc((size_t)nvec * kPoly) || d_r.alloc((size_t)nvec + 1)) return -1;
    if (copy_to_device(d_d.get(), d, (size_t)nvec * kPoly * 4, st)) return -1;
    if (launch_crt_round(d_d.get(), nvec, coef, d_r.get(), st)) return -1;
    HIP_OK(hipMemcpyAsync(r, d_r.get(), (size_t)nvec * 4, hipMemcpyDeviceToHost, st));
    return sync_stream(st);
}

extern "C" int cufe_time_ntt(int npoly, int inverse, int iters, float *ms_per_launch)
{
    Device *dev = device();
    if (!dev) return -1;
    hipStream_t st = dev->stream;
    DevBuf<uint32_t> d;
    if (d.alloc((size_t)npoly * kPoly)) return -1;
    // synthetic residues: any fixed pattern in [0, q0)
    HIP_OK(hipMemsetD32Async((hipDeviceptr_t)d.get(), 65537u, (size_t)npoly * kPoly, st));
    // the reference set's tuned transform shape (tuned on first use)
    const PsetState *ps = pset_state(1);
    if (!ps) return -1;
    for (int w = 0; w < 2; ++w)
        if (ps_ntt(*ps, inverse != 0, d.get(), d.get(), npoly * 3, st)) return -1;
    EventTimer tm(st);
    for (int it = 0; it < iters; ++it)
        if (ps_ntt(*ps, inverse != 0, d.get(), d.get(), npoly * 3, st)) return -1;
    float e = tm.stop();
    if (ms_per_launch) *ms_per_launch = e / (iters > 0 ? iters : 1);
    return sync_stream(st);
}

// nstreams streams of ncalls calls each (sampler which), timed per run.
extern "C" int cufe_time_gauss_calls(int nstreams, int ncalls, int which, int iters, float *ms_per_run)
{
    if (nstreams < 1 || nstreams > 65536 || ncalls < 1 || which < 1 || which > 3) {
        ipfe_set_error("cufe_time_gauss_calls: %d streams x %d calls of S%d", nstreams, ncalls, which);
        return -1;
    }
    Device *dev = device();
    if (!dev) return -1;
    hipStream_t st = dev->stream;
    DevBuf<uint32_t> d;
    if (d.alloc((size_t)nstreams * ncalls * kPoly)) return -1;
    std::vector<StreamReq> reqs;
    for (int t = 0; t < nstreams; ++t) {
        uint8_t key[32];
        for (int i = 0; i < 32; ++i) key[i] = (uint8_t)(i * 7 + 3);
        uint32_t *o = d.get() + (size_t)t * ncalls * kPoly;
        reqs.push_back(make_stream(key, (uint16_t)t, which, ncalls, o, o + kPoly, (long long)kPoly));
    }
    if (run_gauss(reqs, st)) return -1;
    EventTimer tm(st);
    for (int it = 0; it < iters; ++it)
        if (run_gauss(reqs, st)) return -1;
    float e = tm.stop();
    if (ms_per_run) *ms_per_run = e / (iters > 0 ? iters : 1);
    return 0;
}

extern "C" int cufe_time_gauss(int nstreams, int which, int iters, float *ms_per_launch)
{
    Device *dev = device();
    if (!dev) return -1;
    hipStream_t st = dev->stream;
    DevBuf<uint32_t> d;
    if (d.alloc((size_t)nstreams * kPoly)) return -1;
    std::vector<StreamReq> reqs;
    for (int t = 0; t < nstreams; ++t) {
        uint8_t key[32];
        for (int i = 0; i < 32; ++i) key[i] = (uint8_t)(i * 7 + 3);
        reqs.push_back(make_stream(key, (uint16_t)t, which, 1, d.get() + (size_t)t * kPoly, nullptr, 0));
    }
    if (run_gauss(reqs, st)) return -1;
    EventTimer tm(st);
    for (int it = 0; it < iters; ++it)
        if (run_gauss(reqs, st)) return -1;
    float e = tm.stop();
    if (ms_per_launch) *ms_per_launch = e / (iters > 0 ? iters : 1);
    return 0;
}

// ===========================================================================
// Variable-length scheme entry points
// ===========================================================================
static int check_l(int l)
{
    if (l < 0 || l > IPFE_L) {
        ipfe_set_error("vector length l=%d outside [0, %d]", l, IPFE_L);
        return -1;
    }
    return 0;
}

extern "C" int cufe_sife_setup(uint32_t *mpk, uint32_t *msk, const unsigned char seed2[32],
                               const unsigned char seed3[32], int l)
{
    if (check_l(l)) return -1;
    return do_setup(mpk, msk, seed2, seed3, l, nullptr);
}

extern "C" int cufe_sife_encrypt(const uint32_t *m, const uint32_t *mpk, uint32_t *c, const unsigned char seed2[32],
                                 const unsigned char seed3[32], int repeat, int l, int nonce0)
{
    if (check_l(l)) return -1;
    return do_encrypt(m, mpk, c, seed2, seed3, repeat, l, nonce0, nullptr);
}

extern "C" int cufe_sife_keygen(const uint32_t *y, const uint32_t *msk, uint32_t *sk, int repeat, int l)
{
    if (check_l(l)) return -1;
    return do_keygen(y, msk, sk, repeat, l, nullptr);
}

extern "C" int cufe_sife_decrypt(const uint32_t *c, const uint32_t *y, const uint32_t *sk, uint32_t *d, int repeat,
                                 int l)
{
    if (check_l(l)) return -1;
    return do_decrypt(c, y, sk, d, repeat, l, nullptr);
}
