// kfa_tile.hpp -- the tile kernel: compile-time radix schedules on strided lines.
//
// A workgroup owns a tile of TL lines of N points.  Line l = (hi, lo), lo = l % nlo, reads
// element e at in[hi*in_hi + lo*in_lo + e*in_el] and writes it at
// out[hi*out_hi + lo*out_lo + e*out_el].  T threads work on a line.  The first stage reads
// its inputs from HBM into registers, the last one writes its outputs from registers to
// HBM, and only the hand-overs between stages go through LDS (a schedule of K stages
// writes and reads the tile K - 1 times).  Consecutive lanes take consecutive lines at the
// same element, so that wave accesses are contiguous where lines are neighbours in HBM:
//   * column loads and stores: the non-last axes of an N-D array (kiss_fftnd.c:172-177
//     walks the same columns), the first pass of the four-step split;
//   * row loads (ROWS): the first stage alone maps consecutive lanes to consecutive
//     elements of one line, for passes whose input lines are contiguous.
// A thread's line is the lane's for every stage but a ROWS first stage, so a butterfly's
// operands sit TL values apart in LDS and a wave touches TL neighbouring values per
// element: the LDS rows are as free of bank conflicts as the HBM rows are contiguous
// (TilePos).
//
// TWID multiplies element e of line l by W^(lo*e), W = exp(-+2*pi*i/tw_n), on the way out:
// the twiddle step between the two passes of the four-step split (Bailey, "FFTs in
// external or hierarchical memory", 1990):  with n = n1 + N1*n2 and k = k2 + N2*k1,
//   X[k2 + N2*k1] = sum_n1 W_N1^(n1*k1) * W_N^(n1*k2) * sum_n2 x[n1 + N1*n2] W_N2^(n2*k2).
// W^a is hi[a >> 10] * lo[a & 1023] from two small FP64 tables; a thread's outputs share one
// such product and a per-line table of the steps between them in LDS.  The factors and
// the products with the values are FP64, rounded once per output: in float their roundings
// made the split less exact than a single schedule (c2c 10^6 1.80e-7 rel-L2 against 1.74e-7).
// The float path only.
//
// REF is the second pass of a fixed-point line longer than one LDS line, which keeps the
// reference's own stage order: column u of a stage is column lo + L1*u of the full
// transform (L1 = the product of the first pass's radices), so every line reads its own
// rows of the full-length stage tables.  Neighbouring lines read neighbouring rows.
#pragma once

#include "kfa_fast.hpp"

namespace kfa {

struct TileArgs {
    const void *in;
    void *out;
    const void *stw;     // stage table of the schedule (the fast kernels' layout)
    const void *tw_hi;   // TWID: W^(q*1024), q <= tw_n/1024 (FP64)
    const void *tw_lo;   // TWID: W^r, r < 1024 (FP64)
    long long nlines, nlo;
    long long in_hi, in_lo, in_el;
    long long out_hi, out_lo, out_el;
    int xcd_group;       // > 1: tiles g*G .. g*G+G-1 (which share cache lines) run on one XCD
    int l1;              // REF: product of the first pass's radices
};

template <class A, bool INV, int T, class RS, int S>
__device__ __forceinline__ void tile_stage(typename A::store2 *lb, const typename A::store2 *stw, int t)
{
    typedef FastStage<A, INV, T, RS, S, false> F;
    typename F::C v[F::J][F::p];
    F::template gather<false>(v, lb, 1, t, true);
    line_sync<T>();  // every input read before the buffer is overwritten
    F::compute(v, stw, t);
    F::template store<false>(v, lb, 1, t, true);
    line_sync<T>();
}

template <class A, bool INV, int T, class RS, int... S>
__device__ __forceinline__ void tile_stages(std::integer_sequence<int, S...>, typename A::store2 *lb,
                                            const typename A::store2 *stw, int t)
{
    (tile_stage<A, INV, T, RS, S>(lb, stw, t), ...);
}

// Workgroup -> tile.  Workgroups are dealt to the 8 XCDs round-robin; with G tiles sharing
// each cache line, the G tiles of a group go to one XCD back to back, so the line is
// fetched into that XCD's L2 once.  Every round of groups starts one XCD further: with rows
// of a power of two values an XCD would otherwise read the same columns of every row,
// which fall in few of its L2's channels (copying columns of 8 values of a 1024 x 1024
// array, x64: 4.82 against 4.71 TB/s; 64 rows of 256 columns 5.67 against 5.46).
__device__ __forceinline__ long long tile_of_block(long long b, long long ntiles, int G)
{
    const long long full = ntiles / (8LL * G) * (8LL * G);  // complete groups; the tail in order
    if (G <= 1 || b >= full)
        return b;
    const long long x = b % 8, s = b / 8;
    return ((s / G) * 8 + (x + s / G) % 8) * G + s % G;
}

// Line pitch in LDS.  The column phases put lanes ln = 0..TL-1 on neighbouring lines and
// the rest of a wave's lanes on the next elements e0: lane (ln, e0) hits bank pair
// (ln * pitch + e0) mod 32, all different when pitch = N + 32 / TL (mod 32) for TL < 32
// (N + 1, the usual odd pitch, puts lanes (ln, e0) and (ln + 1, e0 - 1) on one bank).
template <int N, int TL>
constexpr int tile_pitch()
{
    return N + (TL < 32 ? 32 / TL : 1);
}

// The kernel streams: what bounds it is the access pattern of its column side.  Measured
// against the form that staged the tile through LDS on both sides of the stages (same
// sizes, alternating runs): 64x96x120 x16 74.3 -> 72.0 us, real 1024x1000 x32 forward and
// inverse 270 -> 263 us; c2c 2^20 x64 474 -> 412 us together with HALF.
//
// HALF hands one component over at a time (real parts, then imaginary parts through the
// same space): half the LDS per line, so twice the lines fit a workgroup.  For lengths whose
// rows would otherwise be shorter than a 128-byte line (8 lines of 8-byte values) that
// is worth the extra barriers: the copy of 1024 rows of 8 columns runs at 4.8 TB/s, of 16
// columns at 5.2-5.4.
//
// What a tile's mapping is made of (template argument MODE of k_tile).
enum { TM_ROWS = 1, TM_TWID = 2, TM_REF = 4, TM_HALF = 8 };

// LDS index of element e of tile line ln.  Column tiles: element rows of TL lines, back to
// back; where such a row of 8-byte values is shorter than the 128 bytes that one LDS access
// of 16 lanes covers (TL < 16), one more row is left free after every G elements, G the
// last stage's even radix: its inputs are G elements apart, and with G + 1 rows between
// them neighbouring butterflies fall in different banks.  (Not for 4-byte slots: the
// padded index needs an address register per access, 77 instead of 63 registers for 1024
// points, and a second workgroup per CU is worth more than the two-way conflict of the
// last gather.)  A ROWS tile is written with lanes along the elements: an odd row of
// TL + 1 values.
template <int TL, int CB, bool ROWS, int G>
struct TilePos {
    static constexpr bool padded = !ROWS && CB >= 8 && TL * CB < 128 && G % 2 == 0;
    static constexpr int row = ROWS ? TL + 1 : TL;
    static constexpr int size(int n) { return (padded ? n + n / G : n) * row; }
    __device__ __forceinline__ static int at(int e, int ln) { return (padded ? e + e / G : e) * row + ln; }
};

template <class A, bool INV, int T, int TL, int MODE, class RS>
struct TileStages {
    typedef typename A::store2 St;
    typedef Ops<A> O;
    typedef Cx<A> C;
    static constexpr int K = RS::K;
    static constexpr bool ROWS = (MODE & TM_ROWS) != 0, HALF = (MODE & TM_HALF) != 0;
    // what LDS holds: whole values, or (HALF) one component of every value at a time
    template <bool H, class X>
    struct Slot {
        typedef typename X::store2 type;
    };
    template <class X>
    struct Slot<true, X> {
        typedef typename X::scalar type;
    };
    typedef typename Slot<HALF, A>::type L;
    typedef TilePos<TL, (int)sizeof(L), ROWS, RS::p(RS::K - 1)> Pos;
    template <int S>
    using Stage = FastStage<A, INV, T, RS, S, false>;

    // stage S's butterflies on v; lo: the line's index (REF)
    template <int S, class V>
    __device__ __forceinline__ static void compute(V &v, const St *stw, int t, int l1, int lo)
    {
        typedef Stage<S> F;
        if constexpr ((MODE & TM_REF) != 0) {
            const typename F::Ent *tab = reinterpret_cast<const typename F::Ent *>(stw);
            const typename F::Ent *rows = tab + (long long)l1 * RS::rows_before(S) + S * RS::rot_len();
            const typename F::Ent *gens = tab + (long long)l1 * (RS::rows_before(K) + RS::gens_before(S)) +
                                          K * RS::rot_len();
            F::template compute_rows<false>(v, rows, rows + (long long)l1 * F::m * F::PR, gens, lo, l1, t);
        } else {
            F::compute(v, stw, t);
        }
    }

    // f(j, r, element) for every input (IN) or output of the thread's stage-S butterflies
    template <int S, bool IN, class Fn>
    __device__ __forceinline__ static void each(int t, Fn f)
    {
        typedef Stage<S> F;
#pragma unroll
        for (int j = 0; j < F::J; ++j) {
            if (!F::live(t, j))
                break;
            const int b = F::bidx(t, j);
            const int u = b / F::P, o = b - (b / F::P) * F::P;
#pragma unroll
            for (int r = 0; r < F::p; ++r)
                f(j, r, IN ? u * F::P * F::p + r * F::P + o : b + r * F::NB);
        }
    }

    // Outputs v of stage S (line lw, thread tw of it) through LDS to the inputs n of stage
    // S + 1 (line ln, thread t).  HALF: real parts first, then the imaginary ones through
    // the same space, so that a tile of twice the lines fits.
    template <int S, class V, class W>
    __device__ __forceinline__ static void hand_over(V &v, W &n, L *buf, int lw, int tw, int ln, int t)
    {
        if constexpr (HALF) {
            each<S, false>(tw, [&](int j, int r, int e) { buf[Pos::at(e, lw)] = v[j][r].r; });
            __syncthreads();
            each<S + 1, true>(t, [&](int j, int r, int e) { n[j][r].r = buf[Pos::at(e, ln)]; });
            __syncthreads();
            each<S, false>(tw, [&](int j, int r, int e) { buf[Pos::at(e, lw)] = v[j][r].i; });
            __syncthreads();
            each<S + 1, true>(t, [&](int j, int r, int e) { n[j][r].i = buf[Pos::at(e, ln)]; });
        } else {
            each<S, false>(tw, [&](int j, int r, int e) { buf[Pos::at(e, lw)] = O::pack(v[j][r]); });
            __syncthreads();
            each<S + 1, true>(t, [&](int j, int r, int e) { n[j][r] = O::load(buf[Pos::at(e, ln)]); });
        }
    }

    // Stages S .. K-1 on v, the inputs of stage S; the last stage's outputs are left in `out`.
    template <int S, class V, class Last>
    __device__ __forceinline__ static void from(V &v, L *buf, const St *stw, int ln, int t, int l1, int lo, Last &out)
    {
        compute<S>(v, stw, t, l1, lo);
        __syncthreads();  // every input read before the tile is overwritten
        if constexpr (S + 1 == K - 1) {
            hand_over<S>(v, out, buf, ln, t, ln, t);
            compute<K - 1>(out, stw, t, l1, lo);
        } else {
            C n[Stage<S + 1>::J][Stage<S + 1>::p];
            hand_over<S>(v, n, buf, ln, t, ln, t);
            from<S + 1>(n, buf, stw, ln, t, l1, lo, out);
        }
    }
};

// Complex FP64 values of the four-step twiddles.
struct Cd {
    double r, i;
};
__device__ __forceinline__ Cd cd_mul(Cd a, Cd b) { return Cd{a.r * b.r - a.i * b.i, a.r * b.i + a.i * b.r}; }
// W^ex from the two tables
__device__ __forceinline__ Cd cd_root(const void *hi, const void *lo, unsigned long long ex)
{
    return cd_mul(reinterpret_cast<const Cd *>(hi)[ex >> 10], reinterpret_cast<const Cd *>(lo)[ex & 1023]);
}
__device__ __forceinline__ Cf cd_apply(Cf v, Cd w)
{
    return Cf{(float)((double)v.r * w.r - (double)v.i * w.i), (float)((double)v.r * w.i + (double)v.i * w.r)};
}

// a / b and a % b, a, b >= 0: 32-bit where the launch allows it (small: nlines < 2^31)
__device__ __forceinline__ void tile_divmod(long long a, long long b, bool small, long long &q, long long &r)
{
    if (small) {
        const unsigned d = (unsigned)a / (unsigned)b;
        q = d;
        r = (unsigned)a - d * (unsigned)b;
    } else {
        q = a / b;
        r = a - q * b;
    }
}

template <class A, bool INV, int T, int TL, int MODE, class RS>
__global__ void __launch_bounds__(T *TL, (MODE & TM_HALF) ? 2 * T * TL / 256 : 1) k_tile(TileArgs a)
{
    typedef typename A::store2 St;
    typedef Ops<A> O;
    typedef Cx<A> C;
    typedef TileStages<A, INV, T, TL, MODE, RS> TS;
    constexpr int N = RS::N(), K = RS::K;
    constexpr bool ROWS = TS::ROWS, TWID = (MODE & TM_TWID) != 0;
    typedef typename TS::template Stage<0> F0;
    typedef typename TS::template Stage<K - 1> FL;
    static_assert(K > 1 || !ROWS, "a one-stage tile has one mapping");
    static_assert(!(TWID && A::fixed), "the four-step twiddle is float");
    // outputs per thread, and the W^(lo*step) between them
    constexpr int IT = FL::J * FL::p;
    __shared__ __align__(16) typename TS::L buf[K > 1 ? TS::Pos::size(N) : 1];
    __shared__ Cd s_step[TWID ? TL * IT : 1];

    const int tid = threadIdx.x;
    const long long ntiles = (a.nlines + TL - 1) / TL;
    const long long l0 = tile_of_block(blockIdx.x, ntiles, a.xcd_group) * TL;
    const int nl = (int)((a.nlines - l0) < TL ? (a.nlines - l0) : TL);
    const bool small = a.nlines < 0x7fffffffLL && a.nlo < 0x7fffffffLL;
    const St *stw = reinterpret_cast<const St *>(__builtin_assume_aligned(a.stw, 16));

    // the thread's line in the column mapping
    const int ln = tid % TL, t = tid / TL;
    const bool ok = ln < nl;
    long long hi, lo;
    tile_divmod(l0 + (ok ? ln : 0), a.nlo, small, hi, lo);

    C out[FL::J][FL::p];
    {   // first stage: HBM -> registers (m == 1: input r of butterfly b is element r*NB + b)
        const int t0 = ROWS ? tid % T : t;
        long long h0 = hi, o0 = lo;
        bool ok0 = ok;
        if constexpr (ROWS) {
            ok0 = tid / T < nl;
            tile_divmod(l0 + (ok0 ? tid / T : 0), a.nlo, small, h0, o0);
        }
        const St *src = reinterpret_cast<const St *>(a.in) + h0 * a.in_hi + o0 * a.in_lo;
        const long long step = (long long)F0::NB * a.in_el;
        C v[F0::J][F0::p];
#pragma unroll
        for (int j = 0; j < F0::J; ++j) {
            const St *p0 = src + (long long)(t0 + j * T) * a.in_el;
            const bool get = ok0 && F0::live(t0, j);
#pragma unroll
            for (int r = 0; r < F0::p; ++r)
                v[j][r] = get ? O::load(p0[r * step]) : O::zero();
        }
        if constexpr (TWID) {
            for (int w = tid; w < TL * IT; w += T * TL) {
                const int l = w % TL, i = w / TL;
                long long h, o;
                tile_divmod(l0 + (l < nl ? l : 0), a.nlo, small, h, o);
                // element jT + q*NB of the thread's first, i = j*p + q (< tw_n: lo < tw_n / N)
                const unsigned long long ex =
                    (unsigned long long)o * (unsigned)((i / FL::p) * T + (i % FL::p) * FL::NB);
                s_step[w] = cd_root(a.tw_hi, a.tw_lo, ex);
            }
        }
        TS::template compute<0>(v, stw, t0, a.l1, (int)o0);
        const int lw = ROWS ? tid / T : ln;
        if constexpr (K == 1) {
#pragma unroll
            for (int j = 0; j < F0::J; ++j)
#pragma unroll
                for (int r = 0; r < F0::p; ++r)
                    out[j][r] = v[j][r];
            if constexpr (TWID)
                __syncthreads();  // the step table
        } else if constexpr (K == 2) {
            TS::template hand_over<0>(v, out, buf, lw, t0, ln, t);
            TS::template compute<1>(out, stw, t, a.l1, (int)lo);
        } else {
            typedef typename TS::template Stage<1> F1;
            C n[F1::J][F1::p];
            TS::template hand_over<0>(v, n, buf, lw, t0, ln, t);
            TS::template from<1>(n, buf, stw, ln, t, a.l1, (int)lo, out);
        }
    }

    if (!ok)
        return;
    St *dst = reinterpret_cast<St *>(a.out) + hi * a.out_hi + lo * a.out_lo;
    const long long step = (long long)FL::NB * a.out_el;
    if constexpr (TWID) {
        const Cd base = cd_root(a.tw_hi, a.tw_lo, (unsigned long long)lo * (unsigned)t);  // (< tw_n)
#pragma unroll
        for (int j = 0; j < FL::J; ++j)
#pragma unroll
            for (int q = 0; q < FL::p; ++q)
                if (FL::live(t, j))
                    out[j][q] = cd_apply(out[j][q], cd_mul(base, s_step[(j * FL::p + q) * TL + ln]));
    }
#pragma unroll
    for (int j = 0; j < FL::J; ++j) {
        if (!FL::live(t, j))
            break;
        St *p0 = dst + (long long)(t + j * T) * a.out_el;
#pragma unroll
        for (int q = 0; q < FL::p; ++q)
            p0[q * step] = O::pack(out[j][q]);
    }
}

}  // namespace kfa
