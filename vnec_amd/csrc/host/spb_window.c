/*
 * spb_window.c — plans of windowed tiles (vnec_win.hip) and, for several
 * right-hand sides, of stream tiles (vnec_spmm.hip): where they run, how large
 * their tiles are, and their layout.
 *
 * A selection mode's pick (spb_tune.c) names a plan shape; where windowed
 * tiles apply they run in place of the kernel it names, over the same matrix
 * with the same arithmetic, and the plan keeps reporting the pick.
 */
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include "spb_internal.h"

/* Runs of consecutive columns: the window's gathers are contiguous loads. */
static int contiguous(const spb_csr *a)
{
    uint64_t v[VNEC_NFEAT_INTS];
    if (vnec_feature_ints_ext((SpB_Matrix)a, v) == SpB_SUCCESS) return v[VF_NEC_LARGE] >= 8 * v[VF_RUNS_LARGE];
    vnec_clear_error();
    return 0;
}

/* Over such columns FP64 64-row slices stream better than windowed tiles from
 * this many nonzeros on (banded and block-diagonal matrices of 16.8M nonzeros:
 * slices 29.9-32.4 us, windowed 31.0-33.1; of 8.9M 19.1 against 17.9, of 13.7M
 * 27.6 against 26.7).  FP32 slices never do (16.8M: 21.7-83 against 19.0-23). */
#define WINDOW_SLICE_NNZ ((int64_t)15 << 20)

/* Pattern slices read no columns at all, but a lane sums its row alone: below
 * this many rows of this length most of the chip idles (27-point stencil, 4k
 * rows: slices 4.4 us, windowed 3.6; 14k 5.5, 3.9; 30k 5.5, 4.5; 29-wide band of
 * 14k rows 5.6, 3.9; but 32k rows of 31: 5.3, 5.3, 47k of 27: 5.6, 5.8, and 32k
 * rows of 17: 4.0, 4.4). */
#define WINDOW_PATTERN_ROWS 30000
#define WINDOW_PATTERN_LEN 20

int vnec_window_applies(const spb_csr *a, const vnec_tuning *t)
{
    if (a->nnz == 0 || t->nrhs > 1) return 0;
    switch (t->variant) {
    case VNEC_VAR_L:
    case VNEC_VAR_C:
    case VNEC_VAR_E:
    case VNEC_VAR_D:
        return 1;
    case VNEC_VAR_S:
        return t->encoding == VNEC_ENC_FP32 || (int64_t)a->nnz < WINDOW_SLICE_NNZ || !contiguous(a);
    case VNEC_VAR_G:
        return (int64_t)a->base.row < WINDOW_PATTERN_ROWS &&
               (int64_t)a->nnz >= WINDOW_PATTERN_LEN * (int64_t)a->base.row;
    default:
        return 0;
    }
}

/* Nonzeros per thread.  Few nonzeros: small tiles, so that there are enough
 * workgroups (R-MAT 14, 0.08M: 4.3 us at 4, 4.7 at 8, 5.9 at 16; 0.39M
 * uniform 4.8 / 5.4 / 6.9; 0.55M R-MAT 6.1 / 5.8 / 6.7; 1.4M R-MAT 9.1 / 9.1 /
 * 8.0; 3.9M 22.7 / 20.4 / 18.4).  Two or three nonzeros a row: as many row
 * sums as window entries in LDS (1.3M over 0.7M rows 16.3 / 18.4 / 17.4).
 * Runs of consecutive columns in FP64: the gathers are cheap and the smaller
 * tiles overlap better (16.8M banded 44.6 / 31.0 / 33.8; FP32 35.5 / 21.9 /
 * 19.0). */
static int window_ipt(const spb_csr *a, int enc)
{
    const int64_t nnz = (int64_t)a->nnz, nr = (int64_t)a->base.row;
    if (nnz < 450000 || nnz < 3 * nr) return 4;
    if (nnz < 1100000) return 8;
    if (enc != VNEC_ENC_FP32 && contiguous(a)) return 8;
    return 16;
}

/* LDS of a workgroup up to which two fit a compute unit. */
#define WINDOW_LDS_TWO (80 * 1024 - 256)

static void window_args(const struct vnec_plan_s *p, const void *x_dev, void *y_dev, vnec_win_args *w)
{
    memset(w, 0, sizeof *w);
    w->desc = p->w_desc;
    w->ntiles = p->ntiles;
    w->entries = p->w_entries;
    w->win = p->w_win;
    w->wbase = p->w_base;
    w->woff = p->w_off;
    w->wv = p->w_val;
    w->whi = p->w_hi;
    w->wlo = p->w_lo;
    w->wl = p->w_rank;
    w->wt = p->w_flags;
    w->rmask = p->w_rmask;
    w->rbase = p->w_rbase;
    if (p->tune.encoding == VNEC_ENC_FP32) {
        w->x32 = (const float *)x_dev;
        w->y32 = (float *)y_dev;
        w->slot32 = (float *)p->carry; /* ntiles doubles hold ntiles floats */
    } else {
        w->x = (const double *)x_dev;
        w->y = (double *)y_dev;
        w->slot = p->carry;
    }
    w->ipt = p->w_ipt;
    w->encoding = p->tune.encoding;
}

void vnec_window_release(struct vnec_plan_s *p)
{
    void **own[] = {(void **)&p->w_val,   (void **)&p->w_hi,    (void **)&p->w_lo,   (void **)&p->w_rank,
                    (void **)&p->w_rbase, (void **)&p->w_flags, (void **)&p->w_rmask, (void **)&p->w_win,
                    (void **)&p->w_base,  (void **)&p->w_desc,  (void **)&p->w_off,   (void **)&p->m_val,
                    (void **)&p->m_slot,  (void **)&p->m_col,   (void **)&p->m_desc,  (void **)&p->m_rbase,
                    (void **)&p->m_nsum,  (void **)&p->m_flags, (void **)&p->m_rmask};
    for (size_t i = 0; i < sizeof own / sizeof own[0]; i++) {
        vnec_free_dev(*own[i]);
        *own[i] = NULL;
    }
}

/* A tile boundary fewer than this many nonzeros into a row moves to the row's
 * start, and the tiles are that much shorter than T: fewer cut rows (a slot
 * that stays empty is not read).  T / 16, or T / 64 where that saves a round
 * of resident workgroups (R-MAT 18, 518 tiles of 7680 against 493 of 8064 on
 * 512 workgroups: 20.3 against 17.8 us; power-law rows 59.0 against 52.9; R-MAT
 * 19 FP32, 794 against 757 on 768: 23.7 against 21.1). */
static int window_snap(int64_t T, int64_t weight, int enc)
{
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
        cus = 256;
    const int64_t wgs = (int64_t)cus * (T <= 4096 ? 4 : enc == VNEC_ENC_FP32 ? 3 : 2);
    const int64_t s16 = T - T / 16, s64 = T - T / 64;
    const int64_t p16 = (weight + s16 - 1) / s16, p64 = (weight + s64 - 1) / s64;
    return (int)((p64 + wgs - 1) / wgs < (p16 + wgs - 1) / wgs ? T / 64 : T / 16);
}

static SpB_Info build_at(struct vnec_plan_s *p, const spb_csr *a, int ipt)
{
    hipStream_t s = vnec_stream();
    const int64_t T = VNEC_WIN_THREADS * (int64_t)ipt, nnz = p->nnz;
    const int enc = p->tune.encoding;
    const int snap = window_snap(T, p->nnz + p->nrows * VNEC_WIN_ROW8 / 8, enc);
    const int64_t weight = nnz + p->nrows * VNEC_WIN_ROW8 / 8, P = (weight + T - snap - 1) / (T - snap);
    const int64_t step = (weight + P - 1) / P; /* equal tiles: no sparse last one */
    const size_t slots = (size_t)(P * T), esz = enc == VNEC_ENC_FP32 ? sizeof(float) : sizeof(double);
    const size_t words = (size_t)(p->nrows / 64 + P + 1), chunks = (size_t)(nnz / 64 + P + 1);
    int64_t bytes = 0;
    p->ntiles = P;
    p->w_threads = VNEC_WIN_THREADS;
    p->w_ipt = ipt;
    p->coords = (int32_t *)vnec_malloc_dev(sizeof(int32_t) * 2 * (size_t)(P + 1), &bytes);
    p->carry = (double *)vnec_malloc_dev(sizeof(double) * (size_t)P, &bytes);
    p->w_desc = (int32_t *)vnec_malloc_dev(sizeof(int32_t) * 8 * (size_t)P, &bytes);
    p->w_win = (int32_t *)vnec_malloc_dev(sizeof(int32_t) * (size_t)nnz, NULL);
    p->w_base = (int32_t *)vnec_malloc_dev(sizeof(int32_t) * chunks, NULL);
    p->w_off = (uint16_t *)vnec_malloc_dev(sizeof(uint16_t) * 64 * chunks, NULL);
    if (enc == VNEC_ENC_FP64) p->w_val = (double *)vnec_malloc_dev(sizeof(double) * slots, &bytes);
    else p->w_hi = (float *)vnec_malloc_dev(sizeof(float) * slots, &bytes);
    if (enc == VNEC_ENC_HILO) p->w_lo = (float *)vnec_malloc_dev(sizeof(float) * slots, &bytes);
    p->w_rank = (uint16_t *)vnec_malloc_dev(sizeof(uint16_t) * slots, &bytes);
    p->w_flags = (uint32_t *)vnec_malloc_dev(sizeof(uint32_t) * (size_t)(P * VNEC_WIN_THREADS), &bytes);
    p->w_rmask = (uint64_t *)vnec_malloc_dev(sizeof(uint64_t) * words, &bytes);
    p->w_rbase = (uint16_t *)vnec_malloc_dev(sizeof(uint16_t) * words, &bytes);
    int32_t *tmp = (int32_t *)vnec_malloc_dev(sizeof(int32_t) * (size_t)(2 * P + 2), NULL);
    uint16_t *lcol = (uint16_t *)vnec_malloc_dev(sizeof(uint16_t) * (size_t)nnz, NULL);
    int32_t *nec = tmp, *nsum = tmp + P, *mx_dev = tmp + 2 * P;
    int32_t mx[2] = {0, 0}; /* LDS entries; whether a tile is wide */
    int32_t *hnec = (int32_t *)malloc(sizeof(int32_t) * (size_t)P);
    SpB_Info rc = p->coords && p->carry && p->w_desc && p->w_win && p->w_base && p->w_off &&
                          (enc == VNEC_ENC_FP64 ? (void *)p->w_val : (void *)p->w_hi) &&
                          (enc != VNEC_ENC_HILO || p->w_lo) && p->w_rank && p->w_flags && p->w_rmask &&
                          p->w_rbase && tmp && lcol
                      ? SpB_SUCCESS : SpB_FAILURE;
    if (rc == SpB_SUCCESS && !hnec) rc = vnec_fail("out of memory");
    if (rc == SpB_SUCCESS)
        rc = vnec_hip_ok(vnec_hip_win_coords(a->d_ptr, p->nrows, nnz, P, VNEC_WIN_ROW8, step, snap, p->coords, s), "window tiles");
    if (rc == SpB_SUCCESS) /* (nsum: scratch for the run counts) */
        rc = vnec_hip_ok(vnec_hip_ecr_tiles_pass1(p->col, p->coords, P, lcol, NULL, p->w_win, nec, nsum, s),
                         "windows");
    if (rc == SpB_SUCCESS) rc = vnec_hip_ok(hipMemsetAsync(mx_dev, 0, sizeof mx, s), "memset");
    if (rc == SpB_SUCCESS)
        rc = vnec_hip_ok(vnec_hip_win_list(p->coords, P, p->w_win, nec, p->w_base, p->w_off, mx_dev + 1, s),
                         "window lists");
    if (rc == SpB_SUCCESS)
        rc = vnec_hip_ok(vnec_hip_win_desc(a->d_ptr, p->nrows, p->coords, P, nec, p->w_desc, s), "window rows");
    if (rc == SpB_SUCCESS)
        rc = vnec_hip_ok(vnec_hip_win_layout(a->d_ptr, a->d_val, lcol, p->coords, P, ipt, enc, p->w_val, p->w_hi,
                                             p->w_lo, p->w_rank, p->w_flags, p->w_rmask, p->w_rbase, nec, nsum,
                                             mx_dev, p->carry, s), "window layout");
    if (rc == SpB_SUCCESS)
        rc = vnec_hip_ok(hipMemcpyAsync(mx, mx_dev, sizeof mx, hipMemcpyDeviceToHost, s), "d2h");
    if (rc == SpB_SUCCESS)
        rc = vnec_hip_ok(hipMemcpyAsync(hnec, nec, sizeof(int32_t) * (size_t)P, hipMemcpyDeviceToHost, s), "d2h");
    if (rc == SpB_SUCCESS) rc = vnec_hip_ok(hipStreamSynchronize(s), "window sync");
    vnec_free_dev(tmp);
    vnec_free_dev(lcol);
    if (rc == SpB_SUCCESS) {
        p->w_window = 0;
        int64_t wide = 0; /* entries of the tiles read from the 32-bit lists */
        for (int64_t t = 0; t < P; t++) {
            p->w_window += hnec[t] & ~VNEC_WIN_WIDE;
            if (hnec[t] & VNEC_WIN_WIDE) wide += hnec[t] & ~VNEC_WIN_WIDE;
        }
        p->w_entries = mx[0];
        p->w_wide = wide;
        if (!mx[1]) {
            vnec_free_dev(p->w_win);
            p->w_win = NULL;
        } else {
            bytes += (int64_t)sizeof(int32_t) * nnz;
        }
        if (mx[1] && p->ncols * (int64_t)esz >= ((int64_t)1 << 32)) { /* 32-bit lists throughout */
            vnec_free_dev(p->w_base);
            vnec_free_dev(p->w_off);
            p->w_base = NULL;
            p->w_off = NULL;
            p->w_wide = p->w_window;
        } else {
            bytes += (int64_t)((sizeof(int32_t) + 64 * sizeof(uint16_t)) * chunks);
        }
        if (ipt > 8 && (size_t)(p->w_entries + 1) * esz > WINDOW_LDS_TWO) {
            /* half the tile, so that two workgroups fit a compute unit */
            vnec_window_release(p);
            vnec_free_dev(p->coords);
            vnec_free_dev(p->carry);
            p->coords = NULL;
            p->carry = NULL;
            free(hnec);
            return build_at(p, a, 8);
        }
        vnec_win_args w;
        window_args(p, NULL, NULL, &w);
        rc = vnec_hip_ok(vnec_hip_win_prepare(&w), "window LDS");
    }
    p->dev_bytes += bytes;
    free(hnec);
    return rc;
}

SpB_Info vnec_window_build(struct vnec_plan_s *p, const spb_csr *a)
{
    return build_at(p, a, window_ipt(a, p->tune.encoding));
}

SpB_Info vnec_window_launch(const struct vnec_plan_s *p, const void *x_dev, void *y_dev, hipStream_t s)
{
    vnec_win_args w;
    window_args(p, x_dev, y_dev, &w);
    return vnec_hip_ok(vnec_hip_spmv_win(&w, s), "window kernel");
}

int64_t vnec_window_bytes(const struct vnec_plan_s *p)
{
    const int enc = p->tune.encoding;
    const int64_t vb = enc == VNEC_ENC_HI || enc == VNEC_ENC_FP32 ? 4 : 8, P = p->ntiles;
    /* values and ranks, the window's columns, the threads' flags, the row
     * masks and the tile descriptors */
    return p->nnz * (vb + 2) + 2 * p->w_window + 2 * p->w_wide + p->w_window / 16 +
           4 * (p->nnz + p->w_ipt - 1) / p->w_ipt + 10 * (p->nrows / 64 + P) + 32 * P;
}

int vnec_plan_windowed(vnec_plan plan)
{
    return plan && plan->magic == SPB_MAGIC_PLAN && (plan->w_threads > 0 || plan->m_run > 0);
}


/* Relabelled columns are measured from this size of x and this many nonzeros
 * on (R-MAT 22 with dense rows, x 32 MiB: 494.9 us plain, 388.7 relabelled
 * with the permutation of x; R-MAT 20, x 8 MiB: 78.4 either way; below, the
 * permutation costs more than the lines it saves: R-MAT 18 17.8 -> 20.7). */
#define WINDOW_RELABEL_X ((int64_t)1 << 21)
#define WINDOW_RELABEL_NNZ ((int64_t)1 << 24)

SpB_Info vnec_window_relabel(spb_csr *a, vnec_tuning *t)
{
    const int64_t nr = (int64_t)a->base.row, nc = (int64_t)a->base.col;
    if ((t->variant != VNEC_VAR_L && t->variant != VNEC_VAR_C) || t->encoding != VNEC_ENC_FP64 || t->nrhs > 1 ||
        8 * nc < WINDOW_RELABEL_X || (int64_t)a->nnz <= WINDOW_RELABEL_NNZ)
        return SpB_SUCCESS;
    const int lanes = (t->lanes == 64 ? 0 : t->lanes) | VNEC_LANES_RELABEL;
    if (!a->window_relabel) {
        double *dx = (double *)vnec_malloc_dev(sizeof(double) * (size_t)nc, NULL);
        double *dy = (double *)vnec_malloc_dev(sizeof(double) * (size_t)nr, NULL);
        SpB_Info rc = dx && dy ? SpB_SUCCESS : SpB_FAILURE;
        if (rc == SpB_SUCCESS) rc = vnec_hip_ok(vnec_hip_zero_f64(dx, nc, vnec_stream()), "zero x");
        double ms[2] = {INFINITY, INFINITY};
        for (int k = 0; rc == SpB_SUCCESS && k < 2; k++) {
            vnec_tuning u = *t;
            if (k) u.lanes = lanes;
            vnec_plan p = NULL;
            if (vnec_plan_build_chosen(&p, (SpB_Matrix)a, &u) != SpB_SUCCESS) {
                if (!k) rc = SpB_FAILURE;
                else vnec_clear_error(); /* not a contender */
                continue;
            }
            rc = vnec_time_plan(p, dx, dy, 20, &ms[k]);
            vnec_plan_free_ext(&p);
        }
        vnec_free_dev(dx);
        vnec_free_dev(dy);
        if (rc != SpB_SUCCESS) return rc;
        a->window_relabel = ms[1] < ms[0] ? 2 : 1;
    }
    if (a->window_relabel == 2) t->lanes = lanes;
    return SpB_SUCCESS;
}

/* ------------------------------------------------ several right-hand sides */
/* With 4 and 8 right-hand sides and this many nonzeros (and weighted rows) a
 * stream is 32 nonzeros long instead of 16 (batch of 28.7M: k = 4 178 us at 16,
 * 170 at 32; k = 8 188, 179; uniform 4.2M: 49.1, 50.2 and 66.2, 66.8; R-MAT 18
 * 35.0, 33.7 and 38.1, 38.5; R-MAT 17, 1.9M: 16.9, 18.2 and 20.7, 20.1).  k = 2
 * takes 8 and k = 16 takes 16 throughout: the batch 157 at 8, 163 at 16 for k =
 * 2; uniform 80.9 at 16, 80.4 at 32 for k = 16. */
#define STREAMS_LONG_RUNS ((int64_t)1 << 23)

int vnec_streams_apply(const spb_csr *a, const vnec_tuning *t)
{
    return a->nnz > 0 && t->variant == VNEC_VAR_L && t->encoding == VNEC_ENC_FP64 &&
           (t->nrhs == 2 || t->nrhs == 4 || t->nrhs == 8 || t->nrhs == 16);
}

/* Eight rows weigh as much as this many nonzeros: a tile's row sums, k to a
 * row, stay within 32 KiB of LDS. */
static int streams_row8(int k) { return k == 16 ? 64 : 32; }

SpB_Info vnec_streams_build(struct vnec_plan_s *p, const spb_csr *a)
{
    hipStream_t s = vnec_stream();
    const int k = p->tune.nrhs, q = k < 8 ? k / 2 : 4, row8 = streams_row8(k);
    const int64_t nnz = p->nnz, weight = nnz + p->nrows * row8 / 8;
    const int run = k == 2 ? 8 : k < 16 && weight >= STREAMS_LONG_RUNS ? 32 : 16;
    const int64_t T = (int64_t)256 / q * run;
    const int snap = (int)(T / 32);
    const int64_t P = (weight + T - snap - 1) / (T - snap), step = (weight + P - 1) / P, words = p->nrows / 64 + P + 1;
    int64_t *acct = &p->dev_bytes;
    p->m_val = (double *)vnec_malloc_dev(sizeof(double) * (size_t)(P * T), acct);
    p->m_col = (int32_t *)vnec_malloc_dev(sizeof(int32_t) * (size_t)(P * T), acct);
    p->m_flags = (uint32_t *)vnec_malloc_dev(sizeof(uint32_t) * 2 * (size_t)(P * (256 / q)), acct);
    p->m_rmask = (uint64_t *)vnec_malloc_dev(sizeof(uint64_t) * (size_t)words, acct);
    p->m_rbase = (int32_t *)vnec_malloc_dev(sizeof(int32_t) * (size_t)words, acct);
    p->m_desc = (int32_t *)vnec_malloc_dev(sizeof(int32_t) * 8 * (size_t)P, acct);
    p->m_nsum = (int32_t *)vnec_malloc_dev(sizeof(int32_t) * (size_t)(P + 1), acct);
    p->m_slot = (double *)vnec_malloc_dev(sizeof(double) * (size_t)(P * k), acct);
    int32_t *co = (int32_t *)vnec_malloc_dev(sizeof(int32_t) * 2 * (size_t)(P + 1), NULL);
    int32_t mx = 0, *mx_dev = p->m_nsum ? p->m_nsum + P : NULL;
    SpB_Info rc = p->m_val && p->m_col && p->m_flags && p->m_rmask && p->m_rbase && p->m_desc && p->m_nsum &&
                          p->m_slot && co
                      ? SpB_SUCCESS : SpB_FAILURE;
    if (rc == SpB_SUCCESS)
        rc = vnec_hip_ok(vnec_hip_win_coords(a->d_ptr, p->nrows, nnz, P, row8, step, snap, co, s), "stream tiles");
    if (rc == SpB_SUCCESS)
        rc = vnec_hip_ok(vnec_hip_win_desc(a->d_ptr, p->nrows, co, P, NULL, p->m_desc, s), "stream rows");
    if (rc == SpB_SUCCESS) rc = vnec_hip_ok(hipMemsetAsync(mx_dev, 0, sizeof mx, s), "memset");
    if (rc == SpB_SUCCESS)
        rc = vnec_hip_ok(vnec_hip_spmm_layout(a->d_ptr, a->d_col, a->d_val, co, P, k, run, p->m_val, p->m_col,
                                              p->m_flags, p->m_rmask, p->m_rbase, p->m_nsum, mx_dev, p->m_slot, s),
                         "stream layout");
    if (rc == SpB_SUCCESS) rc = vnec_hip_ok(hipMemcpyAsync(&mx, mx_dev, sizeof mx, hipMemcpyDeviceToHost, s), "d2h");
    if (rc == SpB_SUCCESS) rc = vnec_hip_ok(hipStreamSynchronize(s), "stream sync");
    vnec_free_dev(co);
    p->m_ntiles = P;
    p->m_run = run;
    p->m_sums = mx;
    return rc;
}

int vnec_streams_run(const struct vnec_plan_s *p, const void *x_dev, const void *y_dev)
{
    return p->m_run > 0 && !(((uintptr_t)x_dev | (uintptr_t)y_dev) & 15);
}

SpB_Info vnec_streams_launch(const struct vnec_plan_s *p, const void *x_dev, void *y_dev, int64_t ldy, hipStream_t s)
{
    vnec_spmm_args m;
    memset(&m, 0, sizeof m);
    m.desc = p->m_desc;
    m.ntiles = p->m_ntiles;
    m.sv = p->m_val;
    m.sc = p->m_col;
    m.sf = p->m_flags;
    m.rmask = p->m_rmask;
    m.rbase = p->m_rbase;
    m.nsum = p->m_nsum;
    m.sums = p->m_sums;
    m.x = (const double *)x_dev;
    m.y = (double *)y_dev;
    m.ldy = ldy;
    m.slot = p->m_slot;
    m.ncols = p->ncols;
    m.k = p->tune.nrhs;
    m.run = p->m_run;
    return vnec_hip_ok(vnec_hip_spmm_tiles(&m, s), "stream kernel");
}

int64_t vnec_streams_bytes(const struct vnec_plan_s *p)
{
    return 12 * p->nnz + 8 * (p->nnz + p->m_run - 1) / p->m_run + 12 * (p->nrows / 64 + p->m_ntiles) +
           36 * p->m_ntiles;
}
