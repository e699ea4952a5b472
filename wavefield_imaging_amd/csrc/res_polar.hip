/*
 * Resident polar (2-D) time loop for gfx950 (MI355X): every step of a shot in
 * one cooperative launch, the wavefield held on the chip.  Tiles, rim exchange
 * and its protocol are res_loop.h's with a stencil half-width of 1.
 *
 * A 460 x 572 polar step is a few hundred nanoseconds of arithmetic; as three
 * launches (step, one-way shell, extraction with the next injection) it took
 * 11 us, here 1.4 us: the exchange and its barriers (13.8 us a step as the
 * four launches without that fusion).
 *
 * A step, per block: the rims arrive (every S steps); the trace row of the
 * step before is extracted (its value is the finished field, before the next
 * injection); a block with sources injects into every node of its image, the
 * margin included, so that neighbours agree; the stencil; the one-way nodes;
 * the sponge.
 *
 * One-way nodes (onewayBC_2D, spher_utils.c:518-563).  A node's rule reads
 * the current field at the node and its inward neighbour, and that
 * neighbour's new value before the boundary; only where the r-high line
 * crosses the two theta lines is that neighbour one whose own rule comes
 * first in the sweep, and its value the final one.  So a chain has at most
 * two levels, inside the tile when the tiles at the high faces own
 * AWEFD_POLAR_FACE nodes (the host picks such a tile; padded r of 63-67, 125-127,
 * 187 and some above 1,680 nodes leave the last tile of both widths, 62 and 60,
 * with fewer, and keep the loop of several launches per step).  The host lists the
 * nodes per block, two a thread: the values before the boundary go to the
 * image, a barrier, the listed nodes are evaluated, a barrier, the final
 * values replace them.  Blocks without such nodes store final values at once.
 *
 * Arithmetic, order and selections are k_spher_step2's and k_spher_shell's
 * (spher_kernels.hip): the same bits.
 */
#include "res_tile.h"

#pragma clang fp contract(off)

namespace {

__device__ __forceinline__ float damped(float v, double f) { return (float)((double)v * f); }

/* depth of a node into the sponge (spongeBC_2D, spher_utils.c:641-690), -1
 * outside the strips */
__device__ __forceinline__ int depth(int ir, int ith, int n1, int n2, int nb)
{
    if (ir < nb || ith < nb) return ir < nb ? nb - ir : nb - ith;
    if (ir > n1 - nb || ith > n2 - nb) return ir > n1 - nb ? ir - (n1 - nb) : ith - (n2 - nb);
    return -1;
}

template <int RX, int S>
__global__ __launch_bounds__(AWEFD_RES_NWAVE * WAVE) void k_polar_res(const awefd_polar_args a)
{
    using T = tile<1, RX, S>;
    constexpr int NTHR = T::NTHR, H = T::H, EXT = T::EXT, ZW = T::ZW, OX = T::OX, ISH = T::ISH, MI = AWEFD_POLAR_ITEMS / NTHR;
    extern __shared__ float img[];                     /* [2][rows + 2][64] */
    __shared__ int s_stop[2];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int lb = xcd_remap(blockIdx.x, a.ntz * a.ntx);
    const int tz = lb % a.ntz, txi = lb / a.ntz;
    const int n1 = a.n1, n2 = a.n2;
    const int z0 = tz * ZW - H, xb = txi * OX - H;     /* node of lane 0 and of image row 0 */
    const int ir = z0 + lane;
    const bool own = lane >= H && lane < WAVE - H && ir < n1;
    const bool zin = ir >= 0 && ir < n1;
    const int x0 = xb + 1 + wv * RX;                   /* first row of the wave */
    if (tid < 2) s_stop[tid] = 0;
    for (int i = tid; i < 2 * ISH; i += NTHR) img[i] = 0.f;
    __syncthreads();

    /* the listed one-way nodes of this thread, marked in the image so that
     * the rows' owners know them */
    const int ob = a.obeg[lb], no = a.obeg[lb + 1] - ob;
    awefd_polar_item it_[MI];
#pragma unroll
    for (int i = 0; i < MI; i++) {
        const int k = tid + i * NTHR;
        it_[i].off = it_[i].noff = it_[i].nnoff = -1;
        if (k < no) {
            it_[i] = a.items[ob + k];
            img[it_[i].off] = 1.f;
        }
    }
    __syncthreads();
    unsigned listed = 0;
#pragma unroll
    for (int j = 0; j < RX; j++) listed |= img[(1 + wv * RX + j) * WAVE + lane] != 0.f ? 1u << j : 0u;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MI; i++)
        if (it_[i].off >= 0) img[it_[i].off] = 0.f;

    const unsigned rowb = (unsigned)a.ld * 4u;
    const rsrc_t rV = mk_rsrc(a.vv, (unsigned)n2 * rowb);
    const unsigned vz = zin ? (unsigned)ir * 4u : OOB;
    const bool rint = ir >= AWEFD_SPHER_NOP && ir < n1 - AWEFD_SPHER_NOP;
    const float *pcp = a.pc + 5 * (zin ? ir : 0);
    const float q0 = pcp[0], q1 = pcp[1], q2 = pcp[2], q3 = pcp[3], q4 = pcp[4];
    const bool zero = a.fsrf && ir > n1 - a.nb;        /* freeSurf_2D (spher_utils.c:745-763) */
    float V[RX], A[RX + 2], B[RX + 2];
    double D[RX];
    unsigned inter = 0;
    bool sp = false;
#pragma unroll
    for (int j = 0; j < RX; j++) {
        const int ith = x0 + j;
        const bool in = ith >= 0 && ith < n2;
        V[j] = bld(rV, in ? vz : OOB, in ? (unsigned)ith * rowb : 0u);
        const int di = in && zin ? depth(ir, ith, n1, n2, a.nb) : -1;
        D[j] = di >= 0 ? a.damp[di] : 1.0;
        sp = sp || __any(di >= 0);
        inter |= rint && ith >= AWEFD_SPHER_NOP && ith < n2 - AWEFD_SPHER_NOP ? 1u << j : 0u;
    }
#pragma unroll
    for (int j = 0; j < RX + 2; j++) A[j] = B[j] = 0.f;

    const u64 *const E0 = a.E, *const E1 = a.E + (long)T::WORDS * a.ntz * a.ntx;   /* words by parity */
    const long me = (long)T::WORDS * (txi * a.ntz + tz);
    exchange<T, 1> xch;
    xch.init(tid, tz, txi, a.ntz, a.ntx);
    const unsigned tag0 = a.tag0;
    const int nt = a.nt;

    /* injection nodes of this block's image, the first of each thread in
     * registers with its first contribution */
    const int sb = a.sbeg[lb], ns = a.sbeg[lb + 1] - sb;
    int so = 0, se0 = 0, se1 = 0;
    float sw = 0.f, sr = 0.f, amp = 0.f;
    if (tid < ns) {
        so = a.snode[2 * (sb + tid)];
        const int node = a.snode[2 * (sb + tid) + 1];
        se0 = a.ibeg[node];
        se1 = a.ibeg[node + 1];
        sw = a.iw[2 * se0];
        sr = a.iw[2 * se0 + 1];
    }
    if (ns > 0) amp = a.wav[0];
    auto inject = [&](float *I, int it) {
        if (tid < ns) {
            float v = I[so], inc = amp * sw;
            inc = inc * sr;
            v = v + inc;
            for (int e = se0 + 1; e < se1; e++) {
                inc = amp * a.iw[2 * e];
                inc = inc * a.iw[2 * e + 1];
                v = v + inc;
            }
            I[so] = v;
        }
        for (int i = tid + NTHR; i < ns; i += NTHR) {
            const int o = a.snode[2 * (sb + i)], node = a.snode[2 * (sb + i) + 1];
            float v = I[o];
            for (int e = a.ibeg[node]; e < a.ibeg[node + 1]; e++) {
                float inc = amp * a.iw[2 * e];
                inc = inc * a.iw[2 * e + 1];
                v = v + inc;
            }
            I[o] = v;
        }
    };

    /* receivers of this block: the first of each thread in registers */
    const int nr = a.nr;
    const int rb = nr > 0 ? a.rbeg[lb] : 0, nrec = nr > 0 ? a.rbeg[lb + 1] - rb : 0;
    int r0 = -1, ro = 0;
    float rw[4] = {0.f, 0.f, 0.f, 0.f};
    if (tid < nrec) {
        r0 = a.ridx[rb + tid];
        ro = (a.rj[3 * r0 + 1] - xb) * WAVE + a.rj[3 * r0] - z0;
#pragma unroll
        for (int q = 0; q < 4; q++) rw[q] = a.rw[8 * r0 + q];
    }
    float *tr = a.tr + r0;
    /* trace row `row` from the finished field I */
    auto extract = [&](const float *I, int row) {
        if (r0 >= 0) {
            float s = 0.f;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float t = I[ro + (q & 1) * WAVE + (q >> 1)] * rw[q];
                s = q == 0 ? t : s + t;
            }
            *tr = s;
            tr += nr;
        }
        for (int i = tid + NTHR; i < nrec; i += NTHR) {
            const int r = a.ridx[rb + i], o = (a.rj[3 * r + 1] - xb) * WAVE + a.rj[3 * r] - z0;
            float s = 0.f;
            for (int q = 0; q < 4; q++) {
                const float t = I[o + (q & 1) * WAVE + (q >> 1)] * a.rw[8 * r + q];
                s = q == 0 ? t : s + t;
            }
            a.tr[(long)row * nr + r] = s;
        }
    };
    __syncthreads();

    int dead = 0;
    /* the rims of image I at step `it` (or, at nt, of the last field) */
    auto rims = [&](float *I, int it, const u64 *words) {
        const unsigned tag = tag0 + (unsigned)it;
        xch.publish((u64 *)words + me, tag, I);
        xch.load(words);
        if (__builtin_expect(!xch.finish(words, tag, I, a), 0)) s_stop[(it / S) & 1] = 1;
        lds_barrier();
        dead = __builtin_amdgcn_readfirstlane(s_stop[(it / S) & 1]);
    };

    /* one step: c <- the image of step it (own rows and one around them), p:
     * the previous field's rows, then the new ones, written to the other
     * image; PAR: the step's parity, XCH: it starts with an exchange */
    auto step = [&]<int PAR, bool XCH>(int it, const u64 *words, float (&c)[RX + 2], float (&p)[RX + 2]) {
        float *const I = img + PAR * ISH, *const N = img + (PAR ^ 1) * ISH, *const Nw = N + (1 + wv * RX) * WAVE + lane;
        /* the next step's amplitude, in flight over this one */
        float na = 0.f;
        if (ns > 0 && it + 1 < nt) na = a.wav[it + 1];
        lds_barrier();
        if (XCH) rims(I, it, words);
        if (it > 0 && nrec > 0) extract(I, it - 1);
        if (ns > 0) {
            lds_barrier();
            inject(I, it);
            lds_barrier();
            amp = na;
        }
        const float *Iw = I + wv * RX * WAVE + lane;
#pragma unroll
        for (int j = 0; j < RX + 2; j++) c[j] = Iw[j * WAVE];
#pragma unroll
        for (int j = 0; j < RX; j++) {
            const float cc = c[1 + j];
            const float cra = (q0 * up1(cc) + q1 * cc) + q2 * dn1(cc);
            const float cth = (q3 * c[j] + q4 * cc) + q3 * c[j + 2];
            const float lap = bits((inter >> j) & 1u ? ~0u : 0u, cra + cth, 0.f);
            float pp = p[1 + j];
            if (sp) pp = damped(pp, D[j]);
            p[1 + j] = (V[j] * lap + 2.f * cc) - pp;
        }
        /* a node's final value from its value before the boundary */
        auto final = [&](int j) {
            float f = p[1 + j];
            if (sp) f = damped(f, D[j]);
            return zero ? 0.f : f;
        };
        if (no == 0) {
            if (S > 1 || own) {
#pragma unroll
                for (int j = 0; j < RX; j++) Nw[j * WAVE] = final(j);
            }
            return;
        }
        if (S > 1 || own) {
#pragma unroll
            for (int j = 0; j < RX; j++) Nw[j * WAVE] = p[1 + j];
        }
        lds_barrier();
        float x[MI];
#pragma unroll
        for (int i = 0; i < MI; i++) {
            const awefd_polar_item &e = it_[i];
            if (e.off < 0) continue;
            float u = N[e.noff];
            if (e.nnoff >= 0) u = I[e.nnoff] + (I[e.noff] - N[e.nnoff]) * e.b2;
            u = I[e.noff] + (I[e.off] - u) * e.b;
            u = damped(u, e.damp);
            x[i] = e.zero ? 0.f : u;
        }
        lds_barrier();
        if (S > 1 || own) {
#pragma unroll
            for (int j = 0; j < RX; j++)
                if (!((listed >> j) & 1u)) Nw[j * WAVE] = final(j);
        }
#pragma unroll
        for (int i = 0; i < MI; i++)
            if (it_[i].off >= 0) N[it_[i].off] = x[i];
    };

    if (S == 1) {
        for (int it = 0; it < nt; it += 2) {
            step.template operator()<0, true>(it, E0, A, B);
            if (__builtin_expect(dead, 0) || it + 1 >= nt) break;
            step.template operator()<1, true>(it + 1, E1, B, A);
            if (__builtin_expect(dead, 0)) break;
        }
    } else {
        for (int it = 0; it < nt; it += 2) {
            step.template operator()<0, true>(it, it & 2 ? E1 : E0, A, B);
            if (__builtin_expect(dead, 0) || it + 1 >= nt) break;
            step.template operator()<1, false>(it + 1, NULL, B, A);
        }
    }
    /* the last trace row, with the margin's nodes of the last field */
    float *const L = img + (nt & 1) * ISH;
    if (!dead) {
        lds_barrier();
        if (nr > 0 && (S == 1 || !(nt & 1))) rims(L, nt, (nt / S) & 1 ? E1 : E0);
    }
    /* a block that gave up tells the others and the host */
    if (dead) {
        if (tid == 0) __hip_atomic_store(a.stop, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        return;
    }
    if (nrec > 0) extract(L, nt - 1);
    /* the last two fields: the newest from the image, the one before from the
     * rows it was computed from */
    const rsrc_t rC = mk_rsrc(a.C, (unsigned)n2 * rowb), rP = mk_rsrc(a.P, (unsigned)n2 * rowb);
    const float *Lw = L + (1 + wv * RX) * WAVE + lane;
    if (nt & 1) {
#pragma unroll
        for (int j = 0; j < RX; j++) B[1 + j] = A[1 + j];
    }
    const unsigned vzo = own ? (unsigned)ir * 4u : OOB;
#pragma unroll
    for (int j = 0; j < RX; j++) {
        const int lr = wv * RX + j;                    /* row of the computed ones */
        const bool in = lr >= EXT && lr < EXT + OX && x0 + j < n2;
        const unsigned s = in ? (unsigned)(x0 + j) * rowb : 0u, v = in ? vzo : OOB;
        bst(rC, v, s, Lw[j * WAVE]);
        bst(rP, v, s, B[1 + j]);
    }
}

template <int RX, int S>
struct kernel {
    static constexpr int NTHR = AWEFD_RES_NWAVE * WAVE;
    static constexpr size_t LDS = sizeof(float) * 2 * (size_t)tile<1, RX, S>::ISH;

    static hipError_t attr()
    {
        if (LDS <= 65536) return hipSuccess;
        return hipFuncSetAttribute((const void *)k_polar_res<RX, S>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)LDS);
    }
    static int launch(const awefd_polar_args *one, int nblk, hipStream_t s)
    {
        const hipError_t e = attr();
        if (e != hipSuccess) return (int)e;
        awefd_polar_args a = *one;
        void *args[] = {&a};
        return (int)hipLaunchCooperativeKernel((const void *)k_polar_res<RX, S>, dim3(nblk), dim3(NTHR), args,
                                               (unsigned)LDS, s);
    }
    static int blocks()
    {
        int nb = 0;
        if (attr() != hipSuccess) return 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, (const void *)k_polar_res<RX, S>, NTHR, LDS) != hipSuccess)
            return 0;
        return nb;
    }
};

/* f<kernel> for a compiled tile (awefd__polar_pick's lists) */
template <class F>
int pick(int rx, int S, F f)
{
#define RX_CASE(n, s) case n: return f(kernel<n, s>());
    if (S == 2) switch (rx) {
        RX_CASE(2, 2) RX_CASE(3, 2) RX_CASE(4, 2) RX_CASE(5, 2) RX_CASE(6, 2) RX_CASE(7, 2)
        RX_CASE(8, 2) RX_CASE(9, 2) RX_CASE(10, 2) RX_CASE(11, 2) RX_CASE(12, 2)
    }
    if (S == 1) switch (rx) {
        RX_CASE(2, 1) RX_CASE(3, 1) RX_CASE(4, 1) RX_CASE(6, 1) RX_CASE(8, 1)
    }
#undef RX_CASE
    return -1;
}

} // namespace

extern "C" int awefd__polar_launch(const awefd_polar_args *a, int nblk, int rx, int S, void *stream)
{
    const int e = pick(rx, S, [&](auto k) { return k.launch(a, nblk, (hipStream_t)stream); });
    return e < 0 ? (int)hipErrorInvalidValue : e;
}

extern "C" int awefd__polar_blocks(int rx, int S)
{
    const int n = pick(rx, S, [&](auto k) { return k.blocks(); });
    return n > 0 ? n : 0;
}
