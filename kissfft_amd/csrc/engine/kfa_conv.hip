// kfa_conv.hip -- fast FIR filtering by overlap-scrap (k_conv in kfa_blue.hpp).
//
// The filter spectrum (N complex FP64, scaled by 1/N) comes from the host layer; the engine
// keeps a device copy per (device, N, impulse response), and the stage tables of an N-point
// schedule once for all of them, and runs every complete block of a call in one launch.
#include <hip/hip_runtime.h>

#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

#include "../kfa_engine.h"
#include "kfa_blue.hpp"
#include "kfa_internal.hpp"

namespace kfa {

typedef std::pair<DevBuf, DevBuf> BufPair;

struct ConvPlan {
    const ConvVariant *v = nullptr;
    BufPair stages;  // forward, inverse
    DevBuf mem_h;
};

// Device plans by the response itself (its samples' bytes): at most 1/2 of the spectrum's, and of a
// real one 1/4, to compare per call, and nothing is copied for the look-up (2^16 samples through
// 1000 taps 23.2 -> 21.2 us, 4000 taps 31.5 -> 27.5).
struct ConvKey {
    int dev, nfft, real;
    std::string taps;
};
struct ConvRef {
    int dev, nfft, real;
    const char *taps;
    size_t bytes;
};
struct ConvLess {
    typedef void is_transparent;
    static ConvRef ref(const ConvKey &k) { return {k.dev, k.nfft, k.real, k.taps.data(), k.taps.size()}; }
    static const ConvRef &ref(const ConvRef &k) { return k; }
    template <class X, class Y>
    bool operator()(const X &x, const Y &y) const
    {
        const ConvRef &a = ref(x), &b = ref(y);
        const auto ka = std::make_tuple(a.dev, a.nfft, a.real, a.bytes), kb = std::make_tuple(b.dev, b.nfft, b.real, b.bytes);
        return ka != kb ? ka < kb : memcmp(a.taps, b.taps, a.bytes) < 0;
    }
};

static std::mutex g_conv_mu;
static std::map<ConvKey, std::shared_ptr<const ConvPlan>, ConvLess> g_conv;
static std::map<std::pair<int, const ConvVariant *>, BufPair> g_conv_stages;  // per device

static int conv_plan(int dev, int nfft, int real, const void *H, const void *h, size_t bytes,
                     std::shared_ptr<const ConvPlan> &out)
{
    std::lock_guard<std::mutex> g(g_conv_mu);
    auto it = g_conv.find(ConvRef{dev, nfft, real, (const char *)h, bytes});
    if (it != g_conv.end()) {
        out = it->second;
        return 0;
    }
    auto cp = std::make_shared<ConvPlan>();
    for (const ConvVariant &v : conv_registry())
        if (v.N == nfft && v.real == real) {  // the first registered of a length
            cp->v = &v;
            break;
        }
    if (!cp->v)
        return fail(-2, "fast convolution: no kernel for block length %d (powers of two 256..8192)", nfft);
    int rc;
    BufPair &st = g_conv_stages[{dev, cp->v}];
    if (!st.first || !st.second) {
        const std::vector<unsigned char> tf = float_twiddles(nfft, 0, nfft, 1), ti = float_twiddles(nfft, 1, nfft, 1);
        const std::vector<int> &rad = cp->v->radices;
        if ((rc = make_stage_table_raw(tf.data(), KFA_F32, nfft, rad, cp->v->tw_pad, 0, st.first)) ||
            (rc = make_stage_table_raw(ti.data(), KFA_F32, nfft, {rad.rbegin(), rad.rend()}, cp->v->tw_pad, 0,
                                       st.second)))
            return rc;
    }
    cp->stages = st;
    if ((rc = dev_upload(H, (size_t)nfft * 16, cp->mem_h)))
        return rc;
    g_conv.emplace(ConvKey{dev, nfft, real, std::string((const char *)h, bytes)}, cp);
    out = cp;
    return 0;
}

// Moves `words` 4-byte words from buf[from ..] to buf[0 ..], the spans overlapping or not: one
// workgroup reads them all before it writes any.  (The host's memmove over the bus took
// about 0.1 us a word: a call of 2^26 samples and 1000 taps 434 -> 250 us, of 228398 samples
// and 239 taps 89 -> 25 us.)
constexpr int kMoveThreads = 1024, kMoveWords = 16 * kMoveThreads;
static __global__ void __launch_bounds__(kMoveThreads) k_move_front(unsigned *buf, long long from, int words)
{
    unsigned v[kMoveWords / kMoveThreads];
#pragma unroll
    for (int k = 0; k < kMoveWords / kMoveThreads; ++k) {
        const int i = threadIdx.x + k * kMoveThreads;
        v[k] = i < words ? buf[from + i] : 0u;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kMoveWords / kMoveThreads; ++k) {
        const int i = threadIdx.x + k * kMoveThreads;
        if (i < words)
            buf[i] = v[k];
    }
}

void conv_release()
{
    std::lock_guard<std::mutex> g(g_conv_mu);
    g_conv.clear();
    g_conv_stages.clear();
}

}  // namespace kfa

using namespace kfa;

extern "C" int kfa_fastfir(int type, int nfft, int real, const void *H, const void *h, long long nh, void *in,
                           void *out, long long nout, long long keep, int *moved, void *stream, int sync)
{
    *moved = 0;
    if (type != KFA_F32)
        return fail(-2, "fast convolution is float only (the reference scales by 1/nfft in float)");
    if (nfft <= 0 || nh <= 0 || nh > nfft || nout < 0 || keep < 0)
        return fail(-2, "fast convolution: bad sizes");
    hipStream_t s;
    int dev;
    int rc = call_begin(stream, &s, &dev);
    if (rc || nout == 0)
        return rc;
    std::shared_ptr<const ConvPlan> cp;
    if ((rc = conv_plan(dev, nfft, real, H, h, (size_t)nh * (real ? 4 : 8), cp)))
        return rc;
    const size_t sb = real ? 4 : 8;
    Operand I, O;
    rc = stage_in(in, sb * (size_t)(nout + nh - 1), s, I);
    if (rc == 0)
        rc = stage_out(out, sb * (size_t)nout, s, O);
    if (rc == 0) {
        ConvArgs a{};
        a.in = I.dev;
        a.out = O.dev;
        a.stw_f = cp->stages.first.get();
        a.stw_i = cp->stages.second.get();
        a.H = cp->mem_h.get();
        a.ngood = nfft - nh + 1;
        a.nin = nout + nh - 1;
        a.nout = nout;
        const long long blocks = (nout + a.ngood - 1) / a.ngood;
        a.nlines = real ? (blocks + 1) / 2 : blocks;
        ++g_launches;
        rc = cp->v->launch(a, s) ? fail(-3, "fast convolution launch failed") : 0;
        const long long words = keep * (long long)(sb / 4);
        if (rc == 0 && !I.staged && words > 0 && words <= kMoveWords) {
            // the samples not used yet go to the front of the caller's device buffer, behind
            // the convolution (from the host each word would cross the bus on its own)
            hipLaunchKernelGGL(k_move_front, dim3(1), dim3(kMoveThreads), 0, s, (unsigned *)I.dev,
                               nout * (long long)(sb / 4), (int)words);
            ++g_launches;
            if (hipGetLastError() != hipSuccess)
                rc = fail(-3, "fast convolution: moving the rest failed");
            else
                *moved = 1;
        }
        if (rc == 0)
            rc = finish_out(O, s);
    }
    release(I);
    release(O);
    return call_end(s, sync || I.staged || O.staged, rc);
}
