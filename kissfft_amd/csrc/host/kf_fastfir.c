/*
 * kf_fastfir.c -- overlap-scrap fast FIR (include/kiss_fastfir.h), the plan and stream
 * bookkeeping of the reference's tools/kiss_fastfir.c:55-246 around one GPU launch per
 * call.
 *
 * Plan (kiss_fastfir.c:65-153): block length nfft, ngood = nfft - nh + 1 good samples per
 * block; the impulse response is rotated left by nh-1 (h[nh-1] first, then zeros, then
 * h[0..nh-2] at the end) so that the wrap-around lands in the block's tail; its spectrum,
 * scaled by 1/length, is computed here in FP64 and kept so.  For the real filter the full
 * complex spectrum of the real response is kept: the GPU filters two real blocks per
 * complex transform.  The GPU's blocks have a length of their own (ff_block).
 */
#include <math.h>
#include <string.h>

#include "kf_internal.h"
#include "kiss_fastfir.h"

struct kiss_fastfir_state {
    size_t nfft;
    size_t ngood;
    size_t nh;
    size_t nblk;      /* points of the GPU's transforms (ff_block) */
    int real;
    double *H;        /* nblk FP64 pairs, spectrum / nblk */
    void *taps;       /* the nh samples of the impulse response */
    void *tmpbuf;     /* nfft samples, the flush block */
};

#ifndef FIXED_POINT
/* in-place radix-2 FFT in FP64, forward, n a power of two; w: room for n doubles */
static void fft_f64(double *re, double *im, size_t n, double *w)
{
    size_t i, j, len, k;
    for (i = 1, j = 0; i < n; ++i) {
        size_t bit = n >> 1;
        for (; j & bit; bit >>= 1)
            j ^= bit;
        j ^= bit;
        if (i < j) {
            double t = re[i];
            re[i] = re[j];
            re[j] = t;
            t = im[i];
            im[i] = im[j];
            im[j] = t;
        }
    }
    for (k = 0; k < n / 2; ++k) {
        const double ang = -2.0 * 3.14159265358979323846264338327 * (double)k / (double)n;
        w[2 * k] = cos(ang);
        w[2 * k + 1] = sin(ang);
    }
    for (len = 2; len <= n; len <<= 1)
        for (i = 0; i < n; i += len)
            for (k = 0; k < len / 2; ++k) {
                const double wr = w[2 * k * (n / len)], wi = w[2 * k * (n / len) + 1];
                const size_t a = i + k, b = i + k + len / 2;
                const double xr = re[b] * wr - im[b] * wi, xi = re[b] * wi + im[b] * wr;
                re[b] = re[a] - xr;
                im[b] = im[a] - xi;
                re[a] += xr;
                im[a] += xi;
            }
}
#endif

#ifndef FIXED_POINT
/* Transform length for a response of nh taps.  A call's output depends on nfft only through
 * its sample count (complete blocks of nfft - nh + 1 good samples), so the GPU takes the
 * length that costs least per good sample: the kernel's time per point of a block (ps),
 * times the points per good sample.  A shorter one within a tenth of the least is taken: its
 * transforms round less.  Measured, 2^25 real samples: 30 taps 67 us with 512 or 1024 points,
 * 74 with 2048; 1000 taps 112 us with 4096 points, 119 with 2048, 107 with 8192. */
static size_t ff_block(size_t nh)
{
    static const struct { size_t n; double ps; } len[] = {{256, 3.7}, {512, 3.4}, {1024, 3.5}, {2048, 4.0},
                                                          {4096, 5.0}, {8192, 5.7}};
    enum { COUNT = sizeof len / sizeof len[0] };
    double cost[COUNT], least = 0;
    size_t i;
    for (i = 0; i < COUNT; ++i) {
        cost[i] = len[i].n < nh ? -1 : len[i].ps * (double)len[i].n / (double)(len[i].n - nh + 1);
        if (cost[i] > 0 && (least == 0 || cost[i] < least))
            least = cost[i];
    }
    for (i = 0; i + 1 < COUNT; ++i)
        if (cost[i] > 0 && cost[i] <= 1.1 * least)
            break;
    return len[i].n;
}
#endif

static kiss_fastfir_cfg ff_alloc(const void *h, size_t nh, int real, size_t *pnfft, void *mem, size_t *lenmem)
{
#ifdef FIXED_POINT
    (void)h;
    (void)nh;
    (void)real;
    (void)pnfft;
    (void)mem;
    (void)lenmem;
    KF_ERROR("kiss_fastfir_alloc: float builds only (the spectrum is scaled by 1/nfft in float)");
    return NULL;
#else
    size_t nfft = pnfft ? *pnfft : 0, nblk, i;
    if (nh < 1)
        return NULL;
    if (nfft == 0) {
        /* next power of two at least 2x the impulse response length, kiss_fastfir.c:77-89 */
        size_t k = nh - 1;
        nfft = 2;
        do {
            nfft <<= 1;
        } while (k >>= 1);
        if (nfft < (real ? 2048u : 1024u))
            nfft = real ? 2048u : 1024u;
    }
    if (pnfft)
        *pnfft = nfft;
    if (nfft < 256 || nfft > 8192 || (nfft & (nfft - 1)) || nh > nfft) {
        KF_ERROR("kiss_fastfir_alloc: block length %zu unsupported (powers of two 256..8192, >= taps)", nfft);
        return NULL;
    }
    nblk = ff_block(nh);
    const size_t samp = real ? sizeof(kiss_fft_scalar) : sizeof(kiss_fft_cpx);
    const size_t need = sizeof(struct kiss_fastfir_state) + 2 * sizeof(double) * nblk + samp * (nh + nfft);
    kiss_fastfir_cfg st = NULL;
    if (lenmem == NULL) {
        st = (kiss_fastfir_cfg)malloc(need);
    } else {
        if (mem && *lenmem >= need)
            st = (kiss_fastfir_cfg)mem;
        *lenmem = need;
    }
    if (!st)
        return NULL;
    st->nfft = nfft;
    st->ngood = nfft - nh + 1;
    st->nh = nh;
    st->nblk = nblk;
    st->real = real;
    st->H = (double *)(st + 1);
    st->taps = (void *)(st->H + 2 * nblk);
    st->tmpbuf = (void *)((char *)st->taps + samp * nh);
    memcpy(st->taps, h, samp * nh);

    double *re = (double *)calloc(nblk, sizeof(double)), *im = (double *)calloc(nblk, sizeof(double));
    double *w = (double *)malloc(nblk * sizeof(double));
    if (!re || !im || !w) {
        free(re);
        free(im);
        free(w);
        if (!lenmem)
            free(st);
        return NULL;
    }
    /* the rotated impulse response, kiss_fastfir.c:137-141 */
    for (i = 0; i < nh; ++i) {
        const size_t at = (i == nh - 1) ? 0 : nblk - nh + 1 + i;
        if (real) {
            re[at] = ((const kiss_fft_scalar *)h)[i];
        } else {
            re[at] = ((const kiss_fft_cpx *)h)[i].r;
            im[at] = ((const kiss_fft_cpx *)h)[i].i;
        }
    }
    fft_f64(re, im, nblk, w);
    for (i = 0; i < nblk; ++i) {
        st->H[2 * i] = re[i] / (double)nblk;
        st->H[2 * i + 1] = im[i] / (double)nblk;
    }
    free(re);
    free(im);
    free(w);
    return st;
#endif
}

/* every complete block of the n samples at in; returns the good samples written.  *moved: the
 * samples after them are at the front of `in` already (rest != 0, device memory) */
static size_t ff_blocks(kiss_fastfir_cfg st, void *in, void *out, size_t n, int rest, int *moved)
{
    *moved = 0;
    if (n < st->nfft)
        return 0;
    const size_t nout = ((n - st->nfft) / st->ngood + 1) * st->ngood;
    if (kfa_fastfir(KF_TYPE, (int)st->nblk, st->real, st->H, st->taps, (long long)st->nh, in, out,
                    (long long)nout, rest ? (long long)(n - nout) : 0, moved, NULL, 1) != 0) {
        KF_ERROR("kiss_fastfir: %s", kfa_last_error());
        return 0;
    }
    return nout;
}

static size_t ff_run(kiss_fastfir_cfg st, void *inbuf, void *outbuf, size_t n_new, size_t *offset)
{
    const size_t samp = st->real ? sizeof(kiss_fft_scalar) : sizeof(kiss_fft_cpx);
    const size_t ntot = n_new + *offset;
    int moved;
    if (n_new == 0) {
        /* flush, kiss_fastfir.c:200-217: complete blocks, then the zero-padded rest */
        size_t done = ff_blocks(st, inbuf, outbuf, ntot, 0, &moved), n = ntot - done, keep;
        char *tmp = (char *)st->tmpbuf;
        memset(tmp, 0, samp * st->nfft);
        memcpy(tmp, (const char *)inbuf + samp * done, samp * n);
        if (ff_blocks(st, tmp, tmp, st->nfft, 0, &moved) == 0)
            return done;
        /* good samples of the padded block that come from real input */
        keep = n + st->ngood > st->nfft ? n + st->ngood - st->nfft : 0;
        memcpy((char *)outbuf + samp * done, tmp, samp * keep);
        return done + keep;
    }
    const size_t nwritten = ff_blocks(st, inbuf, outbuf, ntot, 1, &moved);
    *offset = ntot - nwritten;
    if (!moved)
        memmove(inbuf, (const char *)inbuf + samp * nwritten, samp * *offset);
    return nwritten;
}

kiss_fastfir_cfg kiss_fastfir_alloc_cpx(const kiss_fft_cpx *imp_resp, size_t n_imp_resp, size_t *nfft, void *mem,
                                        size_t *lenmem)
{
    return ff_alloc(imp_resp, n_imp_resp, 0, nfft, mem, lenmem);
}

kiss_fastfir_cfg kiss_fastfir_alloc_real(const kiss_fft_scalar *imp_resp, size_t n_imp_resp, size_t *nfft, void *mem,
                                         size_t *lenmem)
{
    return ff_alloc(imp_resp, n_imp_resp, 1, nfft, mem, lenmem);
}

size_t kiss_fastfir_cpx(kiss_fastfir_cfg cfg, kiss_fft_cpx *inbuf, kiss_fft_cpx *outbuf, size_t n_new, size_t *offset)
{
    if (!cfg || cfg->real || !offset)
        return 0;
    return ff_run(cfg, inbuf, outbuf, n_new, offset);
}

size_t kiss_fastfir_real(kiss_fastfir_cfg cfg, kiss_fft_scalar *inbuf, kiss_fft_scalar *outbuf, size_t n_new,
                         size_t *offset)
{
    if (!cfg || !cfg->real || !offset)
        return 0;
    return ff_run(cfg, inbuf, outbuf, n_new, offset);
}
