/*
 * Misfit gradient of the cartesian 2-D loop with respect to squared slowness
 * (host C).  No counterpart in the reference, whose adj=y mode only injects
 * data backwards in time (MAWEFDcart2Dcpu.c:305-316); this is the adjoint of
 * the discrete forward loop the library runs (adj_kernels.hip).
 *
 * awefd_run_ckpt runs the forward loop in place, as awefd_run_dev does, and
 * copies the (current, previous) pair of fields at steps 0, K, 2K, ... into
 * checkpoint memory.  awefd_adjoint_grad visits the segments last to first:
 * it recomputes the fields of a segment from its checkpoint into K-1 segment
 * buffers (out-of-place steps, so the checkpoint survives and no copies are
 * made) and steps the adjoint backwards through them (four adjoint fields
 * in rotation and the dJ/dV accumulator).  Fields held: 2 ceil(nt/K)
 * checkpoints + K-1 segment buffers + 5.  With K = nt the one segment is the
 * whole run: the forward run stores its fields there and nothing is
 * recomputed.
 */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "awefd_model.h"
#include "res_adj.h"
#include "awefd_setup.h"

#define HIPCHK(call)                                                                        \
    do {                                                                                    \
        hipError_t e_ = (call);                                                             \
        if (e_ != hipSuccess) {                                                             \
            rc = awefd__fail(AWEFD_EHIP, "%s: %s (%s:%d)", #call, hipGetErrorString(e_),    \
                             __FILE__, __LINE__);                                           \
            goto done;                                                                      \
        }                                                                                   \
    } while (0)

typedef struct {
    int K, nck, nt;
    int kept;                 /* K = nt and the run stores every field    */
    unsigned gen;             /* model generation of the checkpoints      */
    int valid;
    float *ck;                /* nck pairs (c_{kK}, c_{kK-1})             */
    float *seg;               /* K-1 fields c_{n0+1} .. c_{n0+K-1}        */
    float *A[4], *gV;         /* alpha fields in rotation, dJ/dV (padded) */
    /* receiver and injection nodes bucketed per adjoint tile column: of the
     * single-grid kernel's tiles, (suffix b) of the batched kernel's and
     * (suffix 2) of the two-step pass's overlapping tiles */
    awefd_inj *rinj, *sinj, *rinjb, *sinjb, *rinj2, *sinj2;
    int *rbeg, *sbeg, *rbegb, *sbegb, *rbeg2, *sbeg2;
    unsigned lists_gen;       /* the model's bgen of the lists            */
    int lists_ok;
    awefd_adj2d_args *d_args; /* device copy of the kernel arguments    */
    float *ones;              /* sponge table of ones (runs without dabc) */
    /* resident adjoint loop (res_adj.hip): its tile, rim words and, per wave,
     * its receiver and injection nodes */
    awefd_res_tile rt;
    awefd_res_buf E;
    unsigned tag;
    awefd_inj *rinjr, *sinjr;
    int *rbegr, *sbegr;
} adj_state;

static void free_lists(adj_state *s)
{
    hipFree(s->rinj); hipFree(s->sinj); hipFree(s->rbeg); hipFree(s->sbeg);
    hipFree(s->rinjb); hipFree(s->sinjb); hipFree(s->rbegb); hipFree(s->sbegb);
    hipFree(s->rinj2); hipFree(s->sinj2); hipFree(s->rbeg2); hipFree(s->sbeg2);
    hipFree(s->rinjr); hipFree(s->sinjr); hipFree(s->rbegr); hipFree(s->sbegr);
    s->rinjr = s->sinjr = NULL;
    s->rbegr = s->sbegr = NULL;
    s->rinj = s->sinj = s->rinjb = s->sinjb = s->rinj2 = s->sinj2 = NULL;
    s->rbeg = s->sbeg = s->rbegb = s->sbegb = s->rbeg2 = s->sbeg2 = NULL;
    s->lists_ok = 0;
}

void awefd__adjoint_free(awefd_model *m)
{
    adj_state *s = m ? m->adj : NULL;
    if (!s) return;
    hipSetDevice(m->dev);
    hipFree(s->ck); hipFree(s->seg);
    hipFree(s->A[0]); hipFree(s->A[1]); hipFree(s->A[2]); hipFree(s->A[3]); hipFree(s->gV); hipFree(s->d_args);
    hipFree(s->ones);
    hipFree(s->E.p);
    free_lists(s);
    free(s);
    m->adj = NULL;
}

void awefd_adjoint_release(awefd_model *m)
{
    awefd__adjoint_free(m);
}

static int min_i(int a, int b)
{
    return a < b ? a : b;
}

/* Interpolation points of a 2-D grid as (node, id, weight) entries bucketed
 * per tile, uploaded to the device.  id is the point index (receivers) or
 * the wavelet column (sources: 0 with expl).  ov = 0: tiles of tz x tx
 * nodes, each node in one; ov = nop: the two-step pass's tiles, whose
 * outputs are (64 - 2 ov) x (tx - 2 ov) nodes and whose extent reaches ov
 * beyond them, each node in every tile whose extent holds it (at most two
 * per axis). */
static int point_buckets(const awefd_model *m, int n, const int *j, const float *w, int same_id, int ntz,
                         int ntx, int tz, int tx, int ov, awefd_inj **d_inj, int **d_beg)
{
    const long cap = (ov ? 16L : 4L) * n;
    const int nbucket = ntz * ntx, sz = 64 - 2 * ov, sx = tx - 2 * ov;
    awefd_inj_key *keys = malloc(sizeof(*keys) * (cap > 0 ? cap : 1));
    awefd_inj *e = malloc(sizeof(*e) * (cap > 0 ? cap : 1));
    int *beg = malloc(sizeof(int) * (nbucket + 1));
    int rc = (!keys || !e || !beg) ? awefd__fail(AWEFD_ENOMEM, "gradient point buckets") : AWEFD_OK;
    long ne = 0;
    if (!rc) {
        for (int a = 0; a < n; a++)
            for (int q = 0; q < 4; q++) {
                awefd_inj en;
                en.z = j[3 * a] + (q & 1);
                en.x = j[3 * a + 1] + ((q >> 1) & 1);
                en.y = 0;
                en.src = same_id ? 0 : a;
                en.w = w[8 * a + q];
                en.w2 = 1.f;
                en.w3 = 1.f;
                if (!ov) {
                    keys[ne].e = en;
                    keys[ne++].bucket = en.z / tz + ntz * (en.x / tx);
                    continue;
                }
                /* tile t's extent: [t s - ov, t s - ov + width) */
                const int vz = en.z + ov - 63, vx = en.x + ov - (tx - 1);
                const int tz0 = vz <= 0 ? 0 : (vz + sz - 1) / sz, tz1 = min_i((en.z + ov) / sz, ntz - 1);
                const int tx0 = vx <= 0 ? 0 : (vx + sx - 1) / sx, tx1 = min_i((en.x + ov) / sx, ntx - 1);
                for (int bx = tx0; bx <= tx1; bx++)
                    for (int bz = tz0; bz <= tz1; bz++) {
                        keys[ne].e = en;
                        keys[ne++].bucket = bz + ntz * bx;
                    }
            }
        awefd_sort_inj(keys, ne, nbucket, e, beg);
        hipError_t er = hipMalloc((void **)d_inj, sizeof(*e) * (ne > 0 ? ne : 1));
        if (er == hipSuccess) er = hipMalloc((void **)d_beg, sizeof(int) * (nbucket + 1));
        if (er == hipSuccess && ne) er = awefd__copy(*d_inj, e, sizeof(*e) * ne, hipMemcpyHostToDevice);
        if (er == hipSuccess)
            er = awefd__copy(*d_beg, beg, sizeof(int) * (nbucket + 1), hipMemcpyHostToDevice);
        if (er != hipSuccess) rc = awefd__fail(AWEFD_EHIP, "gradient point buckets: %s", hipGetErrorString(er));
    }
    free(keys); free(e); free(beg);
    return rc;
}

static int check_model(awefd_model *m, const char *who)
{
    if (!m) return awefd__fail(AWEFD_EINVAL, "%s: NULL model", who);
    if (m->p.kind != AWEFD_CART2D) return awefd__fail(AWEFD_EINVAL, "%s: cartesian 2-D models only", who);
    if (!m->p.cden && m->drho)
        return awefd__fail(AWEFD_EINVAL, "%s: constant density only (cden=y or no density set)", who);
    if (m->p.adj || m->hyb || m->sinc)
        return awefd__fail(AWEFD_EINVAL, "%s: adj=y, hybridbc=y and sinc=y loops have no gradient", who);
    if (!m->model_set || !m->src_set || !m->rec_set || !m->wav_set)
        return awefd__fail(AWEFD_ESTATE, "%s: model not fully set up", who);
    const long need = (long)m->p.nt * (m->p.expl ? 1 : m->ns);
    if (m->nwav < need)
        return awefd__fail(AWEFD_EINVAL, "%s: wavelet has %ld samples, the loop reads %ld", who, m->nwav, need);
    return AWEFD_OK;
}

static int dev_alloc(float **p, size_t bytes)
{
    if (*p) return AWEFD_OK;
    hipError_t e = hipMalloc((void **)p, bytes);
    if (e != hipSuccess) {
        *p = NULL;
        return awefd__fail(AWEFD_ENOMEM, "gradient buffers (%zu bytes): %s", bytes, hipGetErrorString(e));
    }
    return AWEFD_OK;
}

static adj_state *state(const awefd_model *m)
{
    return (adj_state *)m->adj;
}

/* Checkpoint interval when the caller names none (ckpt <= 0): nt, every field
 * kept by the forward run and none recomputed, while at least three quarters
 * of the card's memory stays free beside the n models' fields; else
 * ceil(sqrt(nt)).  Keeping them takes a quarter of a gradient's steps away. */
int awefd__adj_interval(awefd_model *const *ms, int n, int ckpt)
{
    const int nt = ms[0]->p.nt;
    size_t need = 0, fr = 0, total = 0;
    if (ckpt > 0) return ckpt < nt ? ckpt : nt;
    for (int i = 0; i < n; i++) {
        const adj_state *s = state(ms[i]);
        if (!(s && s->K == nt && s->seg)) need += sizeof(float) * (size_t)ms[i]->nalloc * (size_t)(nt + 1);
    }
    if (need == 0) return nt;
    if (hipSetDevice(ms[0]->dev) == hipSuccess && hipMemGetInfo(&fr, &total) == hipSuccess && fr >= need + total / 4 * 3)
        return nt;
    return (int)ceil(sqrt((double)nt));
}

int awefd__adj_ckpt_setup(awefd_model *m, int ckpt)
{
    int rc = check_model(m, "checkpointed run");
    if (rc) return rc;
    const int nt = m->p.nt;
    const int K = awefd__adj_interval(&m, 1, ckpt);
    const int nck = (nt + K - 1) / K;
    if ((size_t)m->nalloc * 4 >= 0x80000000u)
        return awefd__fail(AWEFD_EINVAL, "gradient: field of %ld nodes exceeds 2 GiB", m->nalloc);
    if (hipSetDevice(m->dev) != hipSuccess) return awefd__fail(AWEFD_EHIP, "hipSetDevice");
    adj_state *s = state(m);
    if (!s) {
        s = calloc(1, sizeof *s);
        if (!s) return awefd__fail(AWEFD_ENOMEM, "gradient state");
        m->adj = s;
    }
    s->valid = 0;
    if (s->K != K || s->nck != nck) {
        hipFree(s->ck);
        hipFree(s->seg);
        s->ck = s->seg = NULL;
        s->K = K;
        s->nck = nck;
    }
    s->kept = 0;
    if ((rc = dev_alloc(&s->ck, sizeof(float) * (size_t)m->nalloc * 2 * nck))) return rc;
    /* one segment: the forward run stores its fields, if there is memory */
    s->kept = K == nt && (K == 1 || !dev_alloc(&s->seg, sizeof(float) * (size_t)m->nalloc * (K - 1)));
    const int few = (int)ceil(sqrt((double)nt));
    return s->kept || ckpt > 0 || K < nt || few == nt ? AWEFD_OK : awefd__adj_ckpt_setup(m, few);
}

/* Whether the run set up stores every field; a batch sets it for all its
 * shots together. */
int awefd__adj_kept(const awefd_model *m)
{
    return state(m) && state(m)->kept;
}

void awefd__adj_keep(awefd_model *m, int kept)
{
    state(m)->kept = kept;
}

/* Field n of a run that keeps them all; n = -1: the one before the first. */
static float *kept_field(const adj_state *s, long nalloc, int n)
{
    return n < 0 ? s->ck + nalloc : n == 0 ? s->ck : s->seg + (size_t)(n - 1) * nalloc;
}

/* The last step of a run that kept fields 0 .. nt-1, and the model's field
 * pair as its loop leaves it. */
int awefd__adj_kept_end(awefd_model *m, hipStream_t stream)
{
    const adj_state *s = state(m);
    const int nt = m->p.nt;
    awefd_cart_args a;
    awefd__cart_args(m, &a);
    a.nr = 0;
    a.C = kept_field(s, m->nalloc, nt - 1);
    a.P = kept_field(s, m->nalloc, nt - 2);
    a.Pn = m->dC;
    a.it = nt - 1;
    const int e = awefd_launch_cart_step(&a, m->nop, 2, m->p.sse, 0, stream);
    if (e) return awefd__fail(AWEFD_EHIP, "step %d launch: %s", nt - 1, hipGetErrorString((hipError_t)e));
    const hipError_t he = hipMemcpyAsync(m->dP, a.C, sizeof(float) * (size_t)m->nalloc, hipMemcpyDeviceToDevice, stream);
    if (he != hipSuccess) return awefd__fail(AWEFD_EHIP, "last field: %s", hipGetErrorString(he));
    m->steps_done = nt;
    return AWEFD_OK;
}

/* Traces of a run that kept fields 0 .. nt-1, as many rows a launch as a grid
 * has in y. */
int awefd__adj_kept_traces(awefd_model *m, float *dtr, hipStream_t stream)
{
    const adj_state *s = state(m);
    const int nt = m->p.nt, most = 65535;
    awefd_cart_args a;
    awefd__cart_args(m, &a);
    for (int n = 0; n < nt; n += min_i(most, nt - n)) {
        const float *next = n + 1 < nt ? kept_field(s, m->nalloc, n + 1) : NULL;
        const int e = awefd_launch_cart_traces(&a, kept_field(s, m->nalloc, n), next, m->nalloc, min_i(most, nt - n),
                                               dtr + (size_t)n * a.nr, stream);
        if (e) return awefd__fail(AWEFD_EHIP, "traces: %s", hipGetErrorString((hipError_t)e));
    }
    return AWEFD_OK;
}

/* Forward run that keeps every field: the resident loop where the model takes
 * it, else out-of-place steps and one launch for the traces. */
static int run_kept(awefd_model *m, float *dtr)
{
    adj_state *s = state(m);
    const int nt = m->p.nt;
    int rc = AWEFD_OK, e = awefd_launch_fill(s->ck, 2 * m->nalloc, 0.f, m->stream), done = 0;
    if (e) return awefd__fail(AWEFD_EHIP, "gradient reset: %s", hipGetErrorString((hipError_t)e));
    if (m->res.on && !m->prof && ((rc = awefd__res_run(m, dtr, s->seg, &done)) || done)) return rc;
    awefd_cart_args a;
    awefd__cart_args(m, &a);
    a.nr = 0;
    for (int n = 0; n + 1 < nt; n++) {
        a.C = kept_field(s, m->nalloc, n);
        a.P = kept_field(s, m->nalloc, n - 1);
        a.Pn = kept_field(s, m->nalloc, n + 1);
        a.it = n;
        if ((e = awefd_launch_cart_step(&a, m->nop, 2, m->p.sse, 0, m->stream)))
            return awefd__fail(AWEFD_EHIP, "step %d launch: %s", n, hipGetErrorString((hipError_t)e));
    }
    if ((rc = awefd__adj_kept_end(m, m->stream)) || (rc = awefd__adj_kept_traces(m, dtr, m->stream))) return rc;
    const hipError_t he = hipStreamSynchronize(m->stream);
    return he == hipSuccess ? AWEFD_OK : awefd__fail(AWEFD_EHIP, "forward run: %s", hipGetErrorString(he));
}

float *awefd__adj_ckpt(const awefd_model *m, int k)
{
    return state(m)->ck + (size_t)2 * k * m->nalloc;
}

int awefd__adj_K(const awefd_model *m)
{
    return state(m) ? state(m)->K : 0;
}

void awefd__adj_mark(awefd_model *m)
{
    adj_state *s = state(m);
    s->nt = m->p.nt;
    s->gen = m->gen;
    s->valid = 1;
}

int awefd__adj_ready(const awefd_model *m, const char *who)
{
    int rc = check_model((awefd_model *)m, who);
    if (rc) return rc;
    const adj_state *s = state(m);
    if (!s || !s->valid || s->gen != m->gen || s->nt != m->p.nt)
        return awefd__fail(AWEFD_ESTATE, "%s: no checkpoints of the current model (run with checkpoints first)", who);
    return AWEFD_OK;
}

int awefd_run_ckpt(awefd_model *m, float *d_traces, int ckpt)
{
    int rc = awefd__adj_ckpt_setup(m, ckpt);
    if (rc) return rc;
    const adj_state *s = state(m);
    const int nt = m->p.nt, K = s->K;
    const size_t fb = sizeof(float) * (size_t)m->nalloc;
    awefd_cart_args a;
    if ((rc = awefd__ensure_traces(m))) goto done;
    if (s->kept) {
        if (!(rc = run_kept(m, d_traces ? d_traces : m->d_traces))) awefd__adj_mark(m);
        goto done;
    }
    if ((rc = awefd_reset(m))) goto done;
    awefd__cart_args(m, &a);
    for (int it = 0; it < nt; it++) {
        if (it % K == 0) {
            float *c = awefd__adj_ckpt(m, it / K);
            HIPCHK(hipMemcpyAsync(c, m->dC, fb, hipMemcpyDeviceToDevice, m->stream));
            HIPCHK(hipMemcpyAsync(c + m->nalloc, m->dP, fb, hipMemcpyDeviceToDevice, m->stream));
        }
        a.P = m->dP;
        a.C = m->dC;
        a.it = it;
        a.trow = (d_traces ? d_traces : m->d_traces) + (long)it * m->nr;
        int e = awefd_launch_cart_step(&a, m->nop, 2, m->p.sse, 0, m->stream);
        if (e) {
            rc = awefd__fail(AWEFD_EHIP, "step %d launch: %s", it, hipGetErrorString((hipError_t)e));
            goto done;
        }
        float *t = m->dP;
        m->dP = m->dC;
        m->dC = t;
        m->steps_done = it + 1;
    }
    HIPCHK(hipStreamSynchronize(m->stream));
    awefd__adj_mark(m);
done:
    return rc;
}

/* Tiles of the two-step pass: (64 - 2 nop) x (AWEFD_ADJ2_ROWS - 2 nop)
 * outputs each. */
static void adj2_tiles(const awefd_model *m, int *ntz2, int *ntx2)
{
    const int sz = 64 - 2 * m->nop, sx = AWEFD_ADJ2_ROWS - 2 * m->nop;
    *ntz2 = (m->np[0] + sz - 1) / sz;
    *ntx2 = (m->np[1] + sx - 1) / sx;
}

/* The resident adjoint loop's tile, rim words and point lists, for the models
 * whose forward loop is resident: the fewest rows per wave whose blocks fit
 * one per CU.  rt.on = 0: the loop of one launch per step, also where there is
 * no memory.  (Not for a batch, whose backward pass never runs it.) */
static void resadj_prepare(awefd_model *m, adj_state *s)
{
    static const int list[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 0};
    awefd_res_tile *t = &s->rt;
    int cus = 0;
    if (s->rinjr) return;                      /* the lists of these points */
    if (!s->E.p) {
        t->on = 0;
        if (!m->res.on || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, m->dev) != hipSuccess)
            return;
        for (const int *rx = list; *rx; rx++) {
            awefd__res_tile_of(m, m->nop, *rx, 1, AWEFD_RES_NWAVE, t);
            if (t->on && (long)t->ntz * t->ntx <= cus) break;
            t->on = 0;
        }
        if (!t->on) return;
        const size_t bytes = sizeof(unsigned long long) * 2 * (size_t)t->words * t->ntz * t->ntx;
        s->tag = 1;
        t->on = awefd__resadj_blocks(m->nop, t->rx) >= 1 && !awefd__res_grow(&s->E, bytes) &&
                !awefd_launch_fill(s->E.p, (long)(bytes / sizeof(float)), 0.f, m->stream);
        if (t->on && getenv("AWEFD_VERBOSE"))
            fprintf(stderr, "awefd: resident adjoint: %d x %d blocks of %d waves, %d rows per wave\n", t->ntz, t->ntx,
                    t->nw, t->rx);
    }
    if (!t->on) return;
    const int nw = t->ntx * t->nw;
    if (!point_buckets(m, m->nr, m->h_rj, m->h_rw, 0, t->ntz, nw, t->zw, t->rx, 0, &s->rinjr, &s->rbegr) &&
        !point_buckets(m, m->ns, m->h_sj, m->h_sw, m->p.expl, t->ntz, nw, t->zw, t->rx, 0, &s->sinjr, &s->sbegr))
        return;
    hipFree(s->rinjr); hipFree(s->sinjr); hipFree(s->rbegr); hipFree(s->sbegr);
    s->rinjr = s->sinjr = NULL;
    s->rbegr = s->sbegr = NULL;
    hipFree(s->E.p);                           /* no memory: picked again next time */
    memset(&s->E, 0, sizeof s->E);
    t->on = 0;
}

/* Every backward step of a run that kept its fields, as one launch; *done = 0:
 * not taken, or given up on waiting for a block. */
static int resadj_run(awefd_model *m, adj_state *s, const awefd_adj2d_args *g, int *done)
{
    awefd_resadj_args a;
    int rc;
    *done = 0;
    resadj_prepare(m, s);
    if (!s->rt.on || !m->res.on || awefd__res_flag(m)) return AWEFD_OK;
    memset(&a, 0, sizeof a);
    a.nz = g->nz;
    a.nx = g->nx;
    a.ld = g->ld;
    a.ntz = s->rt.ntz;
    a.ntx = s->rt.ntx;
    a.nt = m->p.nt;
    a.c0f = s->ck;
    a.seg = s->seg;
    a.nal = m->nalloc;
    a.V = g->V;
    a.gV = g->gV;
    a.sp1 = g->sp1;
    a.sp2 = g->sp2;
    a.c0 = g->c0;
    for (int k = 0; k < m->nop; k++) {
        a.cz[k] = g->cz[k];
        a.cx[k] = g->cx[k];
    }
    a.rbeg = s->rbegr;
    a.rinj = s->rinjr;
    a.sbeg = s->sbegr;
    a.sinj = s->sinjr;
    a.res = g->res;
    a.nr = g->nr;
    a.wav = g->wav;
    a.wstride = g->wstride;
    a.E = (unsigned long long *)s->E.p;
    a.stop = m->res.stop;
    awefd__res_wait(&a.wmask, &a.wticks);
    if ((rc = awefd__res_tags(&s->E, &s->tag, a.nt, m->stream, &a.tag0))) return rc;
    const int l = awefd__resadj_launch(&a, a.ntz * a.ntx, m->nop, s->rt.rx, m->stream);
    if (l) {
        (void)hipGetLastError();
        if (awefd__res_broken(l))
            return awefd__fail(AWEFD_EHIP, "resident adjoint: %s", hipGetErrorString((hipError_t)l));
        awefd__res_off(&s->rt.on, "adjoint", hipGetErrorString((hipError_t)l));
        return AWEFD_OK;
    }
    const hipError_t e = hipStreamSynchronize(m->stream);
    if (e != hipSuccess) return awefd__fail(AWEFD_EHIP, "resident adjoint: %s", hipGetErrorString(e));
    *done = *(volatile unsigned *)m->res.stop == 0;
    *m->res.stop = 0;
    if (!*done) awefd__res_off(&s->rt.on, "adjoint", "a block gave up waiting");
    return AWEFD_OK;
}

/* Buffers and point buckets of the backward pass (kept across calls). */
int awefd__adj_prepare(awefd_model *m)
{
    adj_state *s = state(m);
    const size_t fb = sizeof(float) * (size_t)m->nalloc;
    int rc = AWEFD_OK;
    if (hipSetDevice(m->dev) != hipSuccess) return awefd__fail(AWEFD_EHIP, "hipSetDevice");
    if (s->K > 1) rc = dev_alloc(&s->seg, fb * (s->K - 1));
    for (int i = 0; i < 4 && !rc; i++) rc = dev_alloc(&s->A[i], fb);
    if (!rc) rc = dev_alloc(&s->gV, fb);
    if (!rc && !m->p.dabc && !s->ones) {
        const long n = m->np[0] > m->np[1] ? m->np[0] : m->np[1];
        rc = dev_alloc(&s->ones, sizeof(float) * n);
        if (!rc && awefd_launch_fill(s->ones, n, 1.f, m->stream))
            rc = awefd__fail(AWEFD_EHIP, "gradient sponge table");
    }
    if (!rc && !s->d_args) {
        hipError_t e = hipMalloc((void **)&s->d_args, sizeof(awefd_adj2d_args));
        if (e != hipSuccess) rc = awefd__fail(AWEFD_ENOMEM, "gradient arguments: %s", hipGetErrorString(e));
    }
    if (rc) return rc;
    /* the points alone: a new velocity leaves the lists (building six of them
     * for 2,000 receivers is 0.6 ms of host time) */
    if (!s->lists_ok || s->lists_gen != m->bgen) {
        free_lists(s);
        const int ntz = (m->np[0] + 63) / 64, tx = AWEFD_ADJ_TX, txb = AWEFD_ADJ_TXB;
        const int ntx = (m->np[1] + tx - 1) / tx, ntxb = (m->np[1] + txb - 1) / txb;
        int ntz2, ntx2;
        adj2_tiles(m, &ntz2, &ntx2);
        const int ex = m->p.expl;
        if ((rc = point_buckets(m, m->nr, m->h_rj, m->h_rw, 0, ntz, ntx, 64, tx, 0, &s->rinj, &s->rbeg))) return rc;
        if ((rc = point_buckets(m, m->ns, m->h_sj, m->h_sw, ex, ntz, ntx, 64, tx, 0, &s->sinj, &s->sbeg))) return rc;
        if ((rc = point_buckets(m, m->nr, m->h_rj, m->h_rw, 0, ntz, ntxb, 64, txb, 0, &s->rinjb, &s->rbegb))) return rc;
        if ((rc = point_buckets(m, m->ns, m->h_sj, m->h_sw, ex, ntz, ntxb, 64, txb, 0, &s->sinjb, &s->sbegb)))
            return rc;
        if ((rc = point_buckets(m, m->nr, m->h_rj, m->h_rw, 0, ntz2, ntx2, 64, AWEFD_ADJ2_ROWS, m->nop, &s->rinj2,
                                &s->rbeg2)))
            return rc;
        if ((rc = point_buckets(m, m->ns, m->h_sj, m->h_sw, ex, ntz2, ntx2, 64, AWEFD_ADJ2_ROWS, m->nop, &s->sinj2,
                                &s->sbeg2)))
            return rc;
        s->lists_ok = 1;
        s->lists_gen = m->bgen;
    }
    return AWEFD_OK;
}

/* Kernel arguments of the backward pass (after awefd__adj_prepare). */
void awefd__adj_args(const awefd_model *m, const float *d_res, awefd_adj2d_args *g)
{
    const adj_state *s = state(m);
    memset(g, 0, sizeof *g);
    for (int i = 0; i < 4; i++) g->A[i] = s->A[i];
    g->ck = s->ck;
    g->seg = s->seg;
    g->nal = m->nalloc;
    g->K = s->K;
    g->res = d_res;
    g->nr = m->nr;
    g->V = m->dvel;
    g->gV = s->gV;
    g->nz = m->np[0];
    g->nx = m->np[1];
    g->ld = m->ld;
    g->mz = m->p.n[0];
    g->mx = m->p.n[1];
    g->nb = m->nb;
    g->dabc = m->p.dabc;
    g->idt2 = (float)(1.0 / ((double)m->p.dt * m->p.dt));
    g->sp1 = m->p.dabc ? m->dsp[0] : s->ones;
    g->sp2 = m->p.dabc ? m->dsp[1] : s->ones;
    g->c0 = m->c2[0];
    for (int k = 1; k <= m->nop; k++) {
        g->cz[k - 1] = m->c2[k];
        g->cx[k - 1] = m->c2[m->nop + k];
    }
    g->ntz = (m->np[0] + 63) / 64;
    g->ntx = (m->np[1] + AWEFD_ADJ_TX - 1) / AWEFD_ADJ_TX;
    g->nblk = g->ntz * g->ntx;
    g->rbeg = s->rbeg;
    g->rinj = s->rinj;
    g->sbeg = s->sbeg;
    g->sinj = s->sinj;
    g->wav = m->d_wav;
    g->wstride = m->p.expl ? 1 : m->ns;
    adj2_tiles(m, &g->ntz2, &g->ntx2);
    g->nblk2 = g->ntz2 * g->ntx2;
    g->rbeg2 = s->rbeg2;
    g->rinj2 = s->rinj2;
    g->sbeg2 = s->sbeg2;
    g->sinj2 = s->sinj2;
}

/* The same for the batched kernel, whose tiles are 64 x AWEFD_ADJ_TXB. */
void awefd__adj_args_batch(const awefd_model *m, const float *d_res, awefd_adj2d_args *g)
{
    const adj_state *s = state(m);
    awefd__adj_args(m, d_res, g);
    g->ntx = (m->np[1] + AWEFD_ADJ_TXB - 1) / AWEFD_ADJ_TXB;
    g->nblk = g->ntz * g->ntx;
    g->rbeg = s->rbegb;
    g->rinj = s->rinjb;
    g->sbeg = s->sbegb;
    g->sinj = s->sinjb;
}

/* Checkpoint segment bases of the batched recompute. */
void awefd__adj_cart_ckpt(const awefd_model *m, awefd_cart_args *a)
{
    const adj_state *s = state(m);
    a->ck = s->ck;
    a->seg = s->seg;
    a->nal = m->nalloc;
    a->K = s->K;
}

/* The buffers a backward pass starts from zero: alpha_nt, alpha_{nt+1}
 * and dJ/dV (src NULL: fill). */
void awefd__adj_zero_jobs(const awefd_model *m, awefd_copy_job *jobs)
{
    const adj_state *s = state(m);
    const int nt = m->p.nt;
    float *z[3] = {s->A[nt & 3], s->A[(nt + 1) & 3], s->gV};
    for (int i = 0; i < 3; i++) {
        jobs[i].src = NULL;
        jobs[i].dst = z[i];
        jobs[i].n = m->nalloc;
    }
}

int awefd_adjoint_grad(awefd_model *m, const float *d_res, float *d_grad)
{
    int rc = awefd__adj_ready(m, "awefd_adjoint_grad");
    if (rc) return rc;
    if (!d_res || !d_grad) return awefd__fail(AWEFD_EINVAL, "awefd_adjoint_grad: NULL buffer");
    adj_state *s = state(m);
    const int nt = m->p.nt, K = s->K, nck = s->nck;
    awefd_cart_args a;
    awefd_adj2d_args g;
    if ((rc = awefd__adj_prepare(m))) goto done;
    awefd__adj_args(m, d_res, &g);
    HIPCHK(awefd__copy(s->d_args, &g, sizeof g, hipMemcpyHostToDevice));
    int done = 0;
    if (s->kept && (rc = resadj_run(m, s, &g, &done))) goto done;
    if (!done) {
        awefd_copy_job z[3];
        awefd__adj_zero_jobs(m, z);
        for (int i = 0; i < 3; i++) {
            int e = awefd_launch_fill(z[i].dst, z[i].n, 0.f, m->stream);
            if (e) {
                rc = awefd__fail(AWEFD_EHIP, "gradient reset: %s", hipGetErrorString((hipError_t)e));
                goto done;
            }
        }
    }
    /* recompute steps: out of place, no trace extraction */
    awefd__cart_args(m, &a);
    a.nr = 0;
    for (int k = done ? -1 : nck - 1; k >= 0; k--) {
        const int n0 = k * K, n1 = n0 + K < nt ? n0 + K : nt;
        float *ckc = awefd__adj_ckpt(m, k), *ckp = ckc + m->nalloc;
#define FIELD(n) ((n) == n0 ? ckc : s->seg + (size_t)((n) - n0 - 1) * m->nalloc)
        for (int n = n0; n + 1 < n1 && !s->kept; n++) {
            a.C = FIELD(n);
            a.P = n == n0 ? ckp : FIELD(n - 1);
            a.Pn = FIELD(n + 1);
            a.it = n;
            int e = awefd_launch_cart_step(&a, m->nop, 2, m->p.sse, 0, m->stream);
            if (e) {
                rc = awefd__fail(AWEFD_EHIP, "recompute step %d: %s", n, hipGetErrorString((hipError_t)e));
                goto done;
            }
        }
#undef FIELD
        /* (in pairs, as the batch takes them, a 400 x 800 shot's 203 blocks
         * need 22 us a pair against 2 x 7.4) */
        for (int n = n1 - 1; n >= n0; n--) {
            int e = awefd_launch_adj2d_step(&g, n, m->nop, m->stream);
            if (e) {
                rc = awefd__fail(AWEFD_EHIP, "adjoint step %d: %s", n, hipGetErrorString((hipError_t)e));
                goto done;
            }
        }
    }
    {
        int e = awefd_launch_adj2d_chain(&g, s->d_args, 1, d_grad, m->stream);
        if (e) {
            rc = awefd__fail(AWEFD_EHIP, "gradient chain: %s", hipGetErrorString((hipError_t)e));
            goto done;
        }
    }
    HIPCHK(hipStreamSynchronize(m->stream));
done:
    if (rc) hipStreamSynchronize(m->stream);
    return rc;
}
