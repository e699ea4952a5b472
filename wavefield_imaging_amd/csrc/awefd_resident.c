/*
 * Host side of the resident 2-D loop (res_loop.h): which models take it, its
 * tile, its point tables and its launches.
 *
 * A cartesian model takes it when it is 2-D in the SSE order with fdorder up
 * to 8, bilinear points, no hybrid boundary, and a compiled tile whose blocks
 * are at most the CUs: at best 3.9 M padded nodes for fdorder 4 (3.7 M for 8),
 * 0.86 M (0.69 M) with variable density, whose records leave registers for at
 * most 4 rows a wave.  Profiled runs, runs with snapshots and
 * awefd_run_noalloc keep the loop of one launch per step, and so do all runs
 * of a second process on a card, whose cooperative queue has one process at a
 * time.  AWEFD_RESIDENT=0
 * turns it off for the models created after, AWEFD_RES_STEPS=1 or 2 asks for
 * that many steps per exchange.
 */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "awefd_model.h"
#include "awefd_setup.h"

#define HIPCHK(call)                                                                        \
    do {                                                                                    \
        hipError_t e_ = (call);                                                             \
        if (e_ != hipSuccess)                                                               \
            return awefd__fail(AWEFD_EHIP, "%s: %s (%s:%d)", #call, hipGetErrorString(e_),  \
                               __FILE__, __LINE__);                                         \
    } while (0)

/* device memory that grows and is otherwise reused */
int awefd__res_grow(awefd_res_buf *b, size_t bytes)
{
    if (b->cap >= bytes && b->p) return AWEFD_OK;
    hipFree(b->p);
    b->p = NULL;
    b->cap = 0;
    hipError_t e = hipMalloc(&b->p, bytes);
    if (e != hipSuccess) return awefd__fail(AWEFD_ENOMEM, "resident loop: %zu bytes: %s", bytes, hipGetErrorString(e));
    b->cap = bytes;
    return AWEFD_OK;
}

/* The loop this model could take, whatever its grid's size. */
int awefd__res_form(const awefd_model *m)
{
    /* AWEFD_NARROW asks for a tile of the one-launch-per-step kernel */
    const char *e = getenv("AWEFD_RESIDENT");
    if (getenv("AWEFD_NARROW")) return 0;
    return m->p.kind == AWEFD_CART2D && m->p.sse && m->nop <= AWEFD_RES_MAXNOP && !m->hyb && !m->sinc &&
           !(e && atoi(e) == 0);
}

typedef int launch_fn(const awefd_res_args *, int, int, int, int, void *);
typedef int blocks_fn(int, int, int);
static launch_fn *const LAUNCH[AWEFD_RES_MAXNOP] = {awefd__res_launch1, awefd__res_launch2, awefd__res_launch3,
                                                    awefd__res_launch4};
static blocks_fn *const BLOCKS[AWEFD_RES_MAXNOP] = {awefd__res_blocks1, awefd__res_blocks2, awefd__res_blocks3,
                                                    awefd__res_blocks4};

/* A tile of rx rows per wave and S steps per exchange on this grid, for a
 * stencil half-width nop. */
void awefd__res_tile_of(const awefd_model *m, int nop, int rx, int S, int nw, awefd_res_tile *t)
{
    const int H = S * nop;
    t->nw = nw;
    t->rx = rx;
    t->S = S;
    t->zw = 64 - 2 * H;
    t->ox = nw * rx - 2 * (S - 1) * nop;
    t->on = t->ox >= H;
    t->ntz = (m->np[0] + t->zw - 1) / t->zw;
    t->ntx = t->on ? (m->np[1] + t->ox - 1) / t->ox : 0;
    t->words = 2L * ((t->ox * H + 15) / 16 * 16) + 2L * H * 64;
}

/* The compiled tile with the fewest rows per wave whose blocks fit nblk: two
 * steps per exchange up to 6 rows of 16 waves, above (the margin then costs
 * more nodes than the chip has) one and 8 waves. */
void awefd__res_pick(const awefd_model *m, int vd, int nblk, awefd_res_tile *t)
{
    static const int rx2[] = {1, 2, 3, 4, 5, 6, 0}, rx2v[] = {1, 2, 3, 4, 0},
                     rx1[] = {8, 10, 12, 14, 16, 18, 20, 22, 24, 26, 28, 30, 32, 0};
    memset(t, 0, sizeof *t);
    const char *e = getenv("AWEFD_RES_STEPS");
    for (int S = 2; S >= 1; S--) {
        const int *list = S == 1 ? (vd ? rx1 + 13 : rx1) : vd ? rx2v : rx2;
        if (e && atoi(e) != S) continue;
        for (; *list; list++) {
            awefd__res_tile_of(m, m->nop, *list, S, S == 2 ? AWEFD_RES_NWAVE2 : AWEFD_RES_NWAVE, t);
            if (t->on && (long)t->ntz * t->ntx <= nblk) return;
        }
    }
    t->on = 0;
}

int awefd__res_launch(int nop, const awefd_res_tile *t, const awefd_res_args *a, int nblk, int vd, hipStream_t s)
{
    return LAUNCH[nop - 1](a, nblk, t->rx, t->S, vd, s);
}

int awefd__res_blocks(int nop, const awefd_res_tile *t, int vd)
{
    return BLOCKS[nop - 1](t->rx, t->S, vd);
}

/* The flag a block raises when it gives up waiting. */
int awefd__res_flag(awefd_model *m)
{
    awefd_res *r = &m->res;
    if (r->stop) return AWEFD_OK;
    const hipError_t e = hipHostMalloc((void **)&r->stop, sizeof(unsigned), hipHostMallocDefault);
    if (e != hipSuccess) {
        r->stop = NULL;
        return awefd__fail(AWEFD_ENOMEM, "resident loop's flag: %s", hipGetErrorString(e));
    }
    *r->stop = 0;
    return AWEFD_OK;
}

/* Rim words and the flag of the tile picked.  The words are taken by the first
 * run: a shot that only ever runs in a batch needs none (2.6 MB beside 5.6 MB of
 * fields for 500 x 900 nodes; 60 uneven shots held 835 MB instead of 596). */
int awefd__res_buffers(awefd_model *m)
{
    awefd_res *r = &m->res;
    int rc = awefd__res_flag(m);
    if (rc || r->E.p) return rc;
    const size_t eb = sizeof(unsigned long long) * 2 * (size_t)r->t.words * r->t.ntz * r->t.ntx;
    if ((rc = awefd__res_grow(&r->E, eb))) return rc;
    const int e = awefd_launch_fill(r->E.p, (long)(eb / sizeof(float)), 0.f, m->stream);
    if (e) {
        hipFree(r->E.p);
        memset(&r->E, 0, sizeof r->E);
        return awefd__fail(AWEFD_EHIP, "resident rims: %s", hipGetErrorString((hipError_t)e));
    }
    r->tag = 1;
    if (getenv("AWEFD_VERBOSE"))
        fprintf(stderr, "awefd: resident 2-D loop: %d x %d blocks of %d waves, %d rows per wave, %d steps per exchange\n",
                r->t.ntz, r->t.ntx, r->t.nw, r->t.rx, r->t.S);
    return AWEFD_OK;
}

int awefd__res_create(awefd_model *m)
{
    awefd_res *r = &m->res;
    if (!awefd__res_form(m)) return AWEFD_OK;
    int cus = 0, coop = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, m->dev) != hipSuccess ||
        hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, m->dev) != hipSuccess || !coop)
        return AWEFD_OK;
    /* one block per CU; density records may come with the model (cden=n) */
    const int vd = !m->p.cden;
    awefd__res_pick(m, vd, cus, &r->t);
    if (!r->t.on && vd) awefd__res_pick(m, 0, cus, &r->t);
    r->on = r->t.on && awefd__res_blocks(m->nop, &r->t, 0) >= 1;
    awefd__res_prepare(m);
    return AWEFD_OK;
}

void awefd__res_free(awefd_model *m)
{
    awefd_res *r = &m->res;
    hipFree(r->E.p);
    hipFree(r->src.p);
    hipFree(r->rec.p);
    hipFree(r->one.p);
    if (r->stop) hipHostFree(r->stop);
    memset(r, 0, sizeof *r);
}

/* Source entries of every wave of every block: those on the nodes it
 * computes (with S = 2 a node of a margin is in several), in the order of the
 * one sorted list, so entries of a node stay in source order; one upload of
 * both tables. */
int awefd__res_sources(awefd_model *m, const awefd_res_tile *t, awefd_res_buf *out, size_t *inj_off)
{
    awefd_inj *e = NULL;
    int *one = NULL, nbucket;
    long n;
    int rc = awefd__cart_buckets(m, m->np[0], 1, m->np[1], &e, &one, &nbucket, &n);
    if (rc) return rc;
    const int ext = (t->S - 1) * m->nop, nb = t->ntz * t->ntx * t->nw;
    const size_t head = (sizeof(int) * (size_t)(nb + 1) + 15) / 16 * 16;
    char *h = NULL;
    for (int pass = 0; pass < 2 && !rc; pass++) {
        /* pass 0 counts, pass 1 places */
        int *beg = (int *)h, *cnt = NULL;
        if (pass == 0 && !(cnt = calloc((size_t)nb + 1, sizeof(int)))) rc = awefd__fail(AWEFD_ENOMEM, "resident source table");
        for (long i = 0; i < n && !rc; i++)
            for (int bx = (e[i].x - ext > 0 ? (e[i].x - ext) / t->ox : 0); bx <= (e[i].x + ext) / t->ox && bx < t->ntx; bx++)
                for (int bz = (e[i].z - ext > 0 ? (e[i].z - ext) / t->zw : 0); bz <= (e[i].z + ext) / t->zw && bz < t->ntz; bz++) {
                    const int lr = e[i].x - (bx * t->ox - ext);
                    if (lr < 0 || lr >= t->nw * t->rx) continue;
                    const int b = (bz + t->ntz * bx) * t->nw + lr / t->rx;
                    if (pass == 0) cnt[b + 1]++;
                    else ((awefd_inj *)(h + head))[beg[b]++] = e[i];
                }
        if (pass == 0 && !rc) {
            for (int b = 0; b < nb; b++) cnt[b + 1] += cnt[b];
            const size_t bytes = head + sizeof(*e) * (size_t)(cnt[nb] > 0 ? cnt[nb] : 1);
            if (!(h = malloc(bytes))) rc = awefd__fail(AWEFD_ENOMEM, "resident source table");
            if (h) memcpy(h, cnt, sizeof(int) * (size_t)(nb + 1));
        }
        free(cnt);
    }
    if (!rc) {
        int *beg = (int *)h;               /* each start has moved to its end */
        const size_t bytes = head + sizeof(*e) * (size_t)(beg[nb] > 0 ? beg[nb] : 1);
        for (int b = nb; b > 0; b--) beg[b] = beg[b - 1];
        beg[0] = 0;
        rc = awefd__res_grow(out, bytes);
        hipError_t he = rc ? hipSuccess : awefd__copy(out->p, h, bytes, hipMemcpyHostToDevice);
        if (he != hipSuccess) rc = awefd__fail(AWEFD_EHIP, "resident source table: %s", hipGetErrorString(he));
        *inj_off = head;
    }
    free(h);
    free(e);
    free(one);
    return rc;
}

/* Receivers per block, by the block that owns their first corner. */
int awefd__res_receivers(awefd_model *m, const awefd_res_tile *t, awefd_res_buf *out, size_t *idx_off)
{
    const int nr = m->nr, nb = t->ntz * t->ntx;
    int *h = calloc((size_t)nb + 1 + (nr > 0 ? nr : 1), sizeof(int));
    if (!h) return awefd__fail(AWEFD_ENOMEM, "resident receiver table");
    int *idx = h + nb + 1;
#define BLOCK(i) (m->h_rj[3 * (i)] / t->zw + t->ntz * (m->h_rj[3 * (i) + 1] / t->ox))
    for (int i = 0; i < nr; i++) h[BLOCK(i) + 1]++;
    for (int b = 0; b < nb; b++) h[b + 1] += h[b];
    for (int i = 0; i < nr; i++) idx[h[BLOCK(i)]++] = i;
#undef BLOCK
    for (int b = nb; b > 0; b--) h[b] = h[b - 1];
    h[0] = 0;
    const size_t bytes = sizeof(int) * ((size_t)nb + 1 + (nr > 0 ? nr : 1));
    int rc = awefd__res_grow(out, bytes);
    if (!rc) {
        hipError_t he = awefd__copy(out->p, h, bytes, hipMemcpyHostToDevice);
        if (he != hipSuccess) rc = awefd__fail(AWEFD_EHIP, "resident receiver table: %s", hipGetErrorString(he));
    }
    *idx_off = sizeof(int) * ((size_t)nb + 1);
    free(h);
    return rc;
}

/* The tables that a setter made stale and whose points are set. */
static int tables(awefd_model *m)
{
    awefd_res *r = &m->res;
    int rc = AWEFD_OK;
    if (!r->src_ok && (m->inj_rec ? m->h_rj : m->h_sj)) {
        rc = awefd__res_sources(m, &r->t, &r->src, &r->inj_off);
        r->src_ok = !rc;
    }
    if (!rc && !r->rec_ok && m->h_rj) {
        rc = awefd__res_receivers(m, &r->t, &r->rec, &r->idx_off);
        r->rec_ok = !rc;
    }
    return rc;
}

/* Ahead of a run, by awefd_create and the point setters: the flag and the
 * tables; what fails is left to the run, which does without. */
void awefd__res_prepare(awefd_model *m)
{
    if (m->res.on && !awefd__res_flag(m)) (void)tables(m);
}

/* First tag of a run of nt steps over the rims of E: tags only grow, so the
 * words of earlier runs never match; when 32 bits run out, E is cleared. */
int awefd__res_tags(awefd_res_buf *E, unsigned *tag, int nt, hipStream_t s, unsigned *tag0)
{
    if (*tag > 0xffffffffu - (unsigned)nt - 1u) {
        const int e = awefd_launch_fill(E->p, (long)(E->cap / sizeof(float)), 0.f, s);
        if (e) return awefd__fail(AWEFD_EHIP, "resident rims: %s", hipGetErrorString((hipError_t)e));
        *tag = 1;
    }
    *tag0 = *tag;
    *tag += (unsigned)nt + 1u;
    return AWEFD_OK;
}

/* 4 s; AWEFD_RES_WAIT=0 gives up at the first poll that finds a word missing
 * (a test's way to the other loop) */
void awefd__res_wait(unsigned *wmask, long long *wticks)
{
    const char *w = getenv("AWEFD_RES_WAIT");
    const int none = w && atoi(w) == 0;
    *wmask = none ? 0u : 1023u;
    *wticks = none ? -1LL : 400000000LL;
}

void awefd__res_args(const awefd_model *m, const awefd_res_tile *t, const awefd_res_buf *src, size_t inj_off,
                     const awefd_res_buf *rec, size_t idx_off, float *dtr, awefd_res_args *a)
{
    memset(a, 0, sizeof *a);
    a->n1 = m->np[0];
    a->n2 = m->np[1];
    a->ld = m->ld;
    a->ntz = t->ntz;
    a->ntx = t->ntx;
    a->nb = m->nb;
    a->dabc = m->sponge;
    a->c0 = m->c2[0];
    for (int k = 1; k <= m->nop; k++) {
        a->cz[k - 1] = m->c2[k];
        a->cx[k - 1] = m->c2[m->nop + k];
        a->bz[k - 1] = m->c1[k];
        a->bx[k - 1] = m->c1[m->nop + k];
    }
    a->vel = m->dvel;
    a->rho = m->p.cden ? NULL : m->drho;
    a->sp1 = m->dsp[0];
    a->sp2 = m->dsp[1];
    a->P = m->dP;
    a->C = m->dC;
    a->nt = m->nsteps;
    a->ibeg = (const int *)src->p;
    a->inj = (const awefd_inj *)((const char *)src->p + inj_off);
    a->wav = m->p.adj ? m->d_wavr : m->d_wav;
    a->wexpl = m->p.expl;
    a->wstride = m->p.expl ? 1 : m->inj_rec ? m->nr : m->ns;
    a->nr = m->adj2 ? 0 : m->nr;
    a->rbeg = (const int *)rec->p;
    a->ridx = (const int *)((const char *)rec->p + idx_off);
    a->rj = m->d_rj;
    a->rw = m->d_rw;
    a->tr = dtr;
    awefd__res_wait(&a->wmask, &a->wticks);
}

/* Whether a launch error is a failure of the device or of an earlier kernel.
 * Every other one is the cooperative launch's refusal, for which the caller has
 * another loop: too many blocks, not supported, or (hipErrorIllegalState) a
 * second process on a card, one process at a time having its cooperative queue. */
int awefd__res_broken(int e)
{
    return e == hipErrorIllegalAddress || e == hipErrorLaunchFailure || e == hipErrorLaunchTimeOut ||
           e == hipErrorAssert || e == hipErrorECCNotCorrectable || e == hipErrorNoDevice ||
           e == hipErrorInvalidContext || e == hipErrorContextIsDestroyed;
}

/* The resident loop `who` is not tried again by this handle: *on = 0. */
void awefd__res_off(int *on, const char *who, const char *why)
{
    *on = 0;
    if (getenv("AWEFD_VERBOSE")) fprintf(stderr, "awefd: resident %s off: %s\n", who, why);
}

/* After a launch: its wait, and whether every block went through (*done).  A
 * block that gave up waited for 4 s, so that is not tried twice. */
int awefd__res_finish(awefd_model *m, int launched, int *done)
{
    awefd_res *r = &m->res;
    if (launched) {
        (void)hipGetLastError();
        if (awefd__res_broken(launched))
            return awefd__fail(AWEFD_EHIP, "resident loop: %s", hipGetErrorString((hipError_t)launched));
        awefd__res_off(&r->on, "loop", hipGetErrorString((hipError_t)launched));
        return AWEFD_OK;
    }
    HIPCHK(hipStreamSynchronize(m->stream));
    if (*(volatile unsigned *)r->stop) {
        *r->stop = 0;
        awefd__res_off(&r->on, "loop", "a block gave up waiting");
        return AWEFD_OK;
    }
    m->steps_done = m->nsteps;
    *done = 1;
    return AWEFD_OK;
}

/* The whole loop of a set-up model, with its fields 1 .. nt-1 into `fields`
 * (not NULL); *done = 0: not taken (or given up on waiting for a block), the
 * caller runs the other loop from the start. */
int awefd__res_run(awefd_model *m, float *dtr, float *fields, int *done)
{
    awefd_res *r = &m->res;
    awefd_res_args a;
    *done = 0;
    if (!r->on || awefd__res_buffers(m) || tables(m)) return AWEFD_OK;
    awefd__res_args(m, &r->t, &r->src, r->inj_off, &r->rec, r->idx_off, dtr, &a);
    a.F = fields;
    a.nal = m->nalloc;
    const int vd = a.rho != NULL;
    if (vd && awefd__res_blocks(m->nop, &r->t, 1) < 1) return AWEFD_OK;   /* too many rows for the records */
    a.E = (unsigned long long *)r->E.p;
    a.stop = r->stop;
    int rc = awefd__res_tags(&r->E, &r->tag, a.nt, m->stream, &a.tag0);
    if (rc) return rc;
    return awefd__res_finish(m, awefd__res_launch(m->nop, &r->t, &a, r->t.ntz * r->t.ntx, vd, m->stream),
                             done);
}
