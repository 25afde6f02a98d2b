// kfa_blue.hpp -- one-kernel convolutions in LDS: Bluestein's chirp-z transform for float
// lengths with large prime factors, and overlap-scrap fast FIR filtering.
//
// The reference transforms a prime factor p by the direct O(p^2) butterfly
// (kf_bfly_generic, kiss_fft.c:191-233).  For float lines whose schedule contains a large
// prime this kernel computes the same DFT through a cyclic convolution of power-of-two
// length M >= 2N-1 (Bluestein, "A linear filtering approach to the computation of the
// discrete Fourier transform", 1970):
//   w[n] = exp(-+ i*pi*n^2/N),   X[k] = w[k] * sum_n (x[n] w[n]) conj(w[k-n])
// i.e. X = w * IFFT_M( FFT_M(x*w, zero-padded) * B ),  B = FFT_M(conj(w) wrapped) / M.
// One line per T threads, entirely in LDS: the chirp multiply on load, the forward M-point
// schedule, the pointwise product with B, the inverse schedule, the chirp on store.
// w (N entries) and B (M entries) are computed in FP64 on the host; B is rounded once, w as the
// variant asks (CHIRP_*).
#pragma once

#include "kfa_tile.hpp"

namespace kfa {

// ------------------------------------------------------------------------------------
// The cyclic convolution both kernels are made of: x -> IFFT_N(FFT_N(x) * H) on one line of
// N = RS::N() points (a power of two), T threads a line.  The inputs arrive in registers
// as the inputs of the forward schedule's first stage (element r*NB + b of butterfly b),
// the results leave as the outputs of the inverse's last one.  The inverse runs the
// schedule backwards, so its first stage takes exactly the values that the thread's
// forward last stage left, and the product with H happens in registers between the two.
// Only the 2 (K - 1) hand-overs between stages go through LDS.  What bounds the kernels is
// vector arithmetic, then these hand-overs and their barriers.  Against the form that
// staged the line through LDS before, between and after the two transforms (16 trips a
// value with three stages; now 8) and had its inputs 8-way conflicting in LDS banks:
// real FIR of 2^26 samples, 1000 taps (2048-point blocks) 303 -> 250 us (kernel); c2c 1009 x4096
// 36.7 -> 30.9 us (16 values a thread in both).
//
// LDS index of element e: one slot free after every 16, so that the last stage's inputs,
// p = 4 .. 16 elements apart, fall in different banks (N + N/16 slots a line).
// ------------------------------------------------------------------------------------
__device__ __forceinline__ int conv_pos(int e) { return e + (e >> 4); }
constexpr int conv_slots(int n) { return n + n / 16; }

template <class Done, int... X>
struct Reversed;
template <int G, int... Y>
struct Reversed<Radices<G, Y...>> {
    typedef Radices<G, Y...> type;
};
template <int G, int... Y, int X, int... Xs>
struct Reversed<Radices<G, Y...>, X, Xs...> {
    typedef typename Reversed<Radices<G, X, Y...>, Xs...>::type type;
};
template <class RS>
struct Backwards;
template <int G, int R0, int... R>
struct Backwards<Radices<G, R0, R...>> {
    typedef typename Reversed<Radices<G, R0>, R...>::type type;
};

// Stages S .. K-1 of schedule RS on v, the inputs of stage S; the last stage's outputs in
// `out`.  FRESH: the line's LDS holds nothing another thread still reads.  PAIRED: the first
// level of stage S's radix-8 butterflies (which have no twiddles) is done.
template <bool INV, int T, class RS, int S, bool FRESH, bool PAIRED = false, class V, class W>
__device__ __forceinline__ void conv_stages(V &v, W &out, F32::store2 *buf, const F32::store2 *stw, int t)
{
    typedef FastStage<F32, INV, T, RS, S, false> F;
    typedef Ops<F32> O;
    if constexpr (PAIRED) {
        static_assert(F::m == 1 && F::p == 8, "butterflies without twiddles");
#pragma unroll
        for (int j = 0; j < F::J; ++j)
            Dft<8, INV>::tail(v[j]);
    } else {
        F::compute(v, stw, t);
    }
    if constexpr (S == RS::K - 1) {
#pragma unroll
        for (int j = 0; j < F::J; ++j)
#pragma unroll
            for (int q = 0; q < F::p; ++q)
                out[j][q] = v[j][q];
    } else {
        typedef FastStage<F32, INV, T, RS, S + 1, false> Fn;
        static_assert(F::NB % T == 0 && Fn::NB % T == 0, "whole butterflies per thread");
        if constexpr (!FRESH)
            line_sync<T>();
#pragma unroll
        for (int j = 0; j < F::J; ++j)
#pragma unroll
            for (int q = 0; q < F::p; ++q)
                buf[conv_pos(t + j * T + q * F::NB)] = O::pack(v[j][q]);
        line_sync<T>();
        Cf n[Fn::J][Fn::p];
#pragma unroll
        for (int j = 0; j < Fn::J; ++j) {
            const int b = t + j * T, u = b / Fn::P, o = b - u * Fn::P;
#pragma unroll
            for (int r = 0; r < Fn::p; ++r)
                n[j][r] = O::load(buf[conv_pos(u * Fn::P * Fn::p + r * Fn::P + o)]);
        }
        conv_stages<INV, T, RS, S + 1, false>(n, out, buf, stw, t);
    }
}

__device__ __forceinline__ Cf conv_mul(Cf v, float2 h) { return Ops<F32>::cmul(v, Ops<F32>::load(h)); }
__device__ __forceinline__ Cf conv_mul(Cf v, Cd h) { return cd_apply(v, h); }
__device__ __forceinline__ Cd cd_mul(Cf v, Cd h) { return cd_mul(Cd{v.r, v.i}, h); }

// HT: the spectrum's entries, float2 or FP64 (Cd).
template <int T, class RS, class HT>
struct Conv {
    typedef typename Backwards<RS>::type RI;
    typedef FastStage<F32, false, T, RS, 0, false> In;          // layout of the inputs
    typedef FastStage<F32, false, T, RS, RS::K - 1, false> Mid;  // ... of the spectrum
    typedef FastStage<F32, true, T, RI, RS::K - 1, false> Out;   // ... of the results
    static_assert(RS::N() % T == 0 && RS::K > 1, "threads per line must divide the length");
    // FP64 spectrum, 4096 points: the products stay FP64 through the first level of the
    // inverse and are rounded after it, two roundings less, so that 1000 taps are as exact as
    // in blocks of 2048 points (1.73e-7 from FP64, 1.75e-7 without).  It costs 94 registers
    // instead of 78, two workgroups of 512 threads per CU instead of three: 2^26 samples
    // 213 -> 236 us (held to 80 registers the kernel spills).
    static constexpr bool PAIRED = sizeof(HT) == sizeof(Cd) && Mid::p == 8 && RS::N() >= 4096;

    __device__ __forceinline__ static void run(Cf (&v)[In::J][In::p], Cf (&out)[Out::J][Out::p], F32::store2 *buf,
                                               const F32::store2 *stw_f, const F32::store2 *stw_i, const HT *H,
                                               int t)
    {
        Cf m[Mid::J][Mid::p];
        conv_stages<false, T, RS, 0, true>(v, m, buf, stw_f, t);
        // (the inverse's first stage reads element r*NB + b as the forward's last one left it)
        if constexpr (PAIRED) {
#pragma unroll
            for (int j = 0; j < Mid::J; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const HT *h = H + t + j * T + q * Mid::NB;
                    const Cd a = cd_mul(m[j][q], h[0]), b = cd_mul(m[j][q + 4], h[4 * Mid::NB]);
                    m[j][q] = Cf{(float)(a.r + b.r), (float)(a.i + b.i)};
                    m[j][q + 4] = Cf{(float)(a.r - b.r), (float)(a.i - b.i)};
                }
        } else {
#pragma unroll
            for (int j = 0; j < Mid::J; ++j)
#pragma unroll
                for (int q = 0; q < Mid::p; ++q)
                    m[j][q] = conv_mul(m[j][q], H[t + j * T + q * Mid::NB]);
        }
        conv_stages<true, T, RI, 0, false, PAIRED>(m, out, buf, stw_i, t);
    }
};

struct BlueArgs {
    const void *in;
    void *out;
    const void *stw_f, *stw_i;  // stage tables of the M-point schedule, and of it backwards
    const void *chirp;          // w[n], n < N, float2
    const void *chirp_wide;     // the same as the variant's CHIRP asks (null where none does)
    const void *bfft;           // B[m], m < M
    int n;
    long long nlines;
    long long in_hi, in_el, out_hi, out_el;
    int nseg;                   // 0: one buffer (in / out); else segments as in FastArgs
    FastSeg seg[KFA_MAX_SEG];
};

// How the products with the chirp are made (template argument CHIRP):
//   CHIRP_F32   float entries;
//   CHIRP_PAIR  on load, entries of two floats, the value and what float leaves of it: the
//               product is rounded, the table is not;
//   CHIRP_F64   on load and store in FP64, rounded once.
enum { CHIRP_F32 = 0, CHIRP_PAIR = 1, CHIRP_F64 = 2 };

struct ChirpPair {
    float r, i, rest_r, rest_i;
};
__device__ __forceinline__ Cf conv_mul(Cf v, ChirpPair w)
{
    const float r = __builtin_fmaf(v.r, w.rest_r, -(v.i * w.rest_i));
    const float i = __builtin_fmaf(v.r, w.rest_i, v.i * w.rest_r);
    return Cf{__builtin_fmaf(v.r, w.r, __builtin_fmaf(-v.i, w.i, r)), __builtin_fmaf(v.r, w.i, __builtin_fmaf(v.i, w.r, i))};
}

template <int CHIRP>
struct ChirpTable {
    typedef float2 type;
    __device__ __forceinline__ static const type *of(const BlueArgs &a) { return reinterpret_cast<const type *>(a.chirp); }
};
template <>
struct ChirpTable<CHIRP_PAIR> {
    typedef ChirpPair type;
    __device__ __forceinline__ static const type *of(const BlueArgs &a) { return reinterpret_cast<const type *>(a.chirp_wide); }
};
template <>
struct ChirpTable<CHIRP_F64> {
    typedef Cd type;
    __device__ __forceinline__ static const type *of(const BlueArgs &a) { return reinterpret_cast<const type *>(a.chirp_wide); }
};

// The Bluestein body for workgroup `blk` of its launch (see k_fast_body).
template <int T, int LPB, int CHIRP, class RS>
__device__ __forceinline__ void k_blue_body(const BlueArgs &a, long long blk)
{
    typedef F32::store2 St;
    typedef Ops<F32> O;
    typedef Cx<F32> C;
    typedef Conv<T, RS, St> CV;
    typedef typename CV::In In;
    typedef typename CV::Out Out;
    constexpr int M = RS::N();
    extern __shared__ __align__(16) unsigned char kfa_blue_smem[];
    const int line = threadIdx.x / T, t = threadIdx.x - line * T;
    St *buf = reinterpret_cast<St *>(kfa_blue_smem) + line * conv_slots(M);
    const long long gl = blk * LPB + line;
    const bool ok = gl < a.nlines;
    const int n = a.n;
    const auto *chirp_in = ChirpTable<CHIRP>::of(a);
    const auto *chirp_out = ChirpTable<CHIRP == CHIRP_F64 ? CHIRP_F64 : CHIRP_F32>::of(a);

    const St *src;
    St *dst;
    line_base<St>(a, ok ? gl : 0, src, dst);
    C v[In::J][In::p], out[Out::J][Out::p];
#pragma unroll
    for (int j = 0; j < In::J; ++j)
#pragma unroll
        for (int r = 0; r < In::p; ++r) {
            const int i = t + j * T + r * In::NB;
            v[j][r] = (ok && i < n) ? conv_mul(O::load(src[(long long)i * a.in_el]), chirp_in[i]) : O::zero();
        }
    CV::run(v, out, buf, reinterpret_cast<const St *>(a.stw_f), reinterpret_cast<const St *>(a.stw_i),
            reinterpret_cast<const St *>(a.bfft), t);
    if (!ok)
        return;
#pragma unroll
    for (int j = 0; j < Out::J; ++j)
#pragma unroll
        for (int q = 0; q < Out::p; ++q) {
            const int i = t + j * T + q * Out::NB;
            if (i < n)
                dst[(long long)i * a.out_el] = O::pack(conv_mul(out[j][q], chirp_out[i]));
        }
}

template <int T, int LPB, int CHIRP, class RS>
__global__ void __launch_bounds__(T *LPB) k_blue(BlueArgs a)
{
    k_blue_body<T, LPB, CHIRP, RS>(a, blockIdx.x);
}

}  // namespace kfa

namespace kfa {

// Fast convolution by overlap-scrap (the reference's tools/kiss_fastfir.c:167-239): block
// k reads the window in[k*ngood .. k*ngood + N), is transformed, multiplied by the filter
// spectrum H (already scaled by 1/N), transformed back, and its first ngood samples --
// the ones the rotated impulse response leaves free of wrap-around -- are written to
// out[k*ngood ..].  The last block may reach past the nin input samples (read as zeros) and
// the nout output samples (not written).  One block per T threads.  REAL: the samples are
// real and two consecutive blocks travel as the real and imaginary parts of one complex
// block; with a real impulse response the two convolutions stay separate.
struct ConvArgs {
    const void *in;
    void *out;
    const void *stw_f, *stw_i;  // stage tables of the N-point schedule, and of it backwards
    const void *H;              // N complex FP64: the product is rounded once, which makes up for
                                // the roundings of a longer block (4096 for 2048 points)
    long long nlines;           // complex blocks (REAL: two blocks of samples each)
    long long ngood;            // samples a block yields
    long long nin, nout;
};

template <int T, int LPB, bool REAL, class RS>
__global__ void __launch_bounds__(T *LPB) k_conv(ConvArgs a)
{
    typedef F32::store2 St;
    typedef Ops<F32> O;
    typedef Cx<F32> C;
    typedef Conv<T, RS, Cd> CV;
    typedef typename CV::In In;
    typedef typename CV::Out Out;
    constexpr int N = RS::N();
    extern __shared__ __align__(16) unsigned char kfa_conv_smem[];
    const int line = threadIdx.x / T, t = threadIdx.x - line * T;
    St *buf = reinterpret_cast<St *>(kfa_conv_smem) + line * conv_slots(N);
    const long long gl = (long long)blockIdx.x * LPB + line;
    const bool ok = gl < a.nlines;
    // the line's first sample, its second block's (REAL), and what is left of the input there
    const long long s0 = (REAL ? 2 * gl : gl) * a.ngood, s1 = s0 + a.ngood;
    auto left = [](long long end, long long at) {
        const long long d = end - at;
        return (int)(d < 0 ? 0 : d < N ? d : N);
    };
    const int in0 = ok ? left(a.nin, s0) : 0, in1 = ok && REAL ? left(a.nin, s1) : 0;

    C v[In::J][In::p], out[Out::J][Out::p];
    if constexpr (REAL) {
        const float *x = reinterpret_cast<const float *>(a.in) + (ok ? s0 : 0);
#pragma unroll
        for (int j = 0; j < In::J; ++j)
#pragma unroll
            for (int r = 0; r < In::p; ++r) {
                const int i = t + j * T + r * In::NB;
                v[j][r] = C{i < in0 ? x[i] : 0.0f, i < in1 ? x[a.ngood + i] : 0.0f};
            }
    } else {
        const St *x = reinterpret_cast<const St *>(a.in) + (ok ? s0 : 0);
#pragma unroll
        for (int j = 0; j < In::J; ++j)
#pragma unroll
            for (int r = 0; r < In::p; ++r) {
                const int i = t + j * T + r * In::NB;
                v[j][r] = i < in0 ? O::load(x[i]) : O::zero();
            }
    }
    CV::run(v, out, buf, reinterpret_cast<const St *>(a.stw_f), reinterpret_cast<const St *>(a.stw_i),
            reinterpret_cast<const Cd *>(a.H), t);
    if (!ok)
        return;
    const int good = (int)a.ngood, out0 = left(a.nout, s0), out1 = REAL ? left(a.nout, s1) : 0;
#pragma unroll
    for (int j = 0; j < Out::J; ++j)
#pragma unroll
        for (int q = 0; q < Out::p; ++q) {
            const int i = t + j * T + q * Out::NB;
            if (i >= good)
                continue;
            if constexpr (REAL) {
                float *y = reinterpret_cast<float *>(a.out) + s0;
                if (i < out0)
                    y[i] = out[j][q].r;
                if (i < out1)
                    y[good + i] = out[j][q].i;
            } else if (i < out0) {
                (reinterpret_cast<St *>(a.out) + s0)[i] = O::pack(out[j][q]);
            }
        }
}

}  // namespace kfa
