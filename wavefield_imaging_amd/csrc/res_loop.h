/*
 * Resident cartesian 2-D time loop for gfx950 (MI355X): every step of a shot
 * in one launch, the wavefield held on the chip.  Included by one source
 * file per stencil half-width (RES_NOP).
 *
 * A 2-D grid of this program is a few hundred thousand nodes; the chip has
 * 128 MB of vector registers and 40 MB of LDS.  One launch per step leaves
 * the time to the launches (a 500 x 900 step is 0.1 us of arithmetic per
 * SIMD in a 3.7 us kernel), larger grids to 16 bytes per node and step from
 * the Infinity Cache.  Here each block owns a tile for the whole loop: the
 * previous field and (v dt)^2 of its nodes stay in registers, the current
 * field in LDS, and only the rim of the tile goes through device memory to
 * the neighbouring blocks, once every S steps.
 *
 * Rim exchange.  A rim value travels as one 64-bit word {tag, value}, stored
 * and polled with device-scope relaxed atomics (8 bytes, so value and tag
 * arrive together: no separate flag and no fence; the poll's own wait covers
 * the stores issued before it, which share its counter).
 * Alone, one exchange between 8 to 256 blocks takes 0.75-0.95 us (64 words a
 * side), whichever XCDs the neighbours sit on.  Words are double-buffered by
 * the parity of the exchange: a block overwrites exchange e's words at
 * e + 2, after it has the words e + 1 of every block that reads its own,
 * which they send only after reading its e; so reading is mutual, the
 * diagonal neighbours included.  Tags grow over the life of the buffer
 * (awefd_resident.c), so no word needs clearing between runs.  The rim is
 * stored in whole 64-word groups, one wave each, after a barrier: when each
 * wave stored the words of its own rows, several waves shared a 128-byte
 * line, and a line takes one partial write at a time (8 waves of 1 row:
 * 1.2 us a step).
 *
 * S steps per exchange: the tile carries a margin of S NOP nodes on every
 * side; each step consumes NOP of it, and the blocks compute the margin's
 * inner nodes redundantly.  S = 2 halves the exchanges for a margin of 2 NOP
 * nodes a side instead of NOP (S NOP in general, (S - 1) NOP of them
 * computed); the chip holds fewer owned nodes, so the largest grids run S = 1.
 * More than two steps an exchange were not built.
 *
 * Progress.  The launch is cooperative: all blocks are resident before any
 * runs.  A wait is bounded all the same: after 4 s without its words (or
 * once another block has given up) a block raises the stop flag and leaves;
 * the host then runs the one-launch-per-step loop instead, from then on for
 * that handle.
 *
 * Tile.  A wave holds 64 z lanes, the outer S NOP on each side the margin,
 * of RX x rows; 16 waves a block with S = 2 (4 per SIMD, up to 96 rows: the
 * waves' chains of dependent steps overlap; 8 waves of twice the rows took
 * 1.47 us a step for 140 x 240 nodes against 1.24, 1.49 against 1.30 for
 * 500 x 900, 2.5 against 2.3 for 800 x 1500), 8 with S = 1, whose rows need
 * the registers (28 rows as 16 waves of 14: 13.4 us against 9.5).  z neighbours are DPP shifts inside the
 * wave, x neighbours rows of the block's LDS image, which also feeds the
 * trace extraction (a receiver belongs to the block of its first corner; the
 * other corners are in the margin).  The image is double-buffered by the
 * parity of the step.
 *
 * Measured per step, against one launch per step: 140 x 240 nodes 1.24 us
 * (3.1 as a graph), 500 x 900 1.30 us (4.7 launched, 3.66 as a graph), 1101 x
 * 2877 with nop 4 8.2 us (11.2).  What a step takes at the small sizes: the
 * exchange 0.6 us per step with S = 2 (1.0 with S = 1: 2.3 and 2.0 us in
 * all), barriers and LDS rows 0.3, arithmetic 0.1-0.3; at 30 rows per wave
 * the arithmetic about 4 us and the exchange of 2,300 words a block 3.5 (the
 * even row counts matter there: 32 rows of which 30 were needed took 9.4).
 *
 * Arithmetic, order and selections are cart_step_body's (cart_kernels.hip)
 * node for node, lazy second sponge included: the same bits.
 */
#include "res_tile.h"

#pragma clang fp contract(off)

namespace {

typedef const awefd_res_args __attribute__((address_space(4))) cargs;

/* entries before this lane's (of m in lanes) on the same node */
__device__ __forceinline__ int node_rank(const awefd_inj &en, int lane, int m)
{
    int rank = 0;
    for (int e = 0; e + 1 < m; e++) {
        const int ex = __builtin_amdgcn_readlane(en.x, e), ez = __builtin_amdgcn_readlane(en.z, e);
        rank += e < lane && ex == en.x && ez == en.z ? 1 : 0;
    }
    return lane < m ? rank : -1;
}

/* ((amp w) w2) w3 v added to the nodes of a wave's entries, entries of one
 * node one after the other; row0: the image at the wave's first row, lane 0
 * being node z0 */
__device__ __forceinline__ void inject(const cargs &a, awefd_inj en, int rank, float amp, float v, int ib,
                                       int ne, int lane, int it, float *row0, int x0, int z0)
{
    for (int e0 = 0;;) {
        const float q = amp * en.w * en.w2 * en.w3;
        for (int k = 0; __any(rank >= k); k++)
            if (rank == k) {
                float *const u = row0 + (en.x - x0) * WAVE + en.z - z0;
                *u = *u + q * v;
            }
        e0 += WAVE;
        if (e0 >= ne) break;
        const int m = ne - e0 < WAVE ? ne - e0 : WAVE;
        if (lane < m) {
            en = a.inj[ib + e0 + lane];
            amp = a.wav[(long)it * a.wstride + (a.wexpl ? 0 : en.src)];
            v = a.vel[(long)en.x * a.ld + en.z];
        }
        rank = node_rank(en, lane, m);
    }
}

template <int NOP>
struct coef {
    float c0, cz[NOP], cx[NOP], bz[NOP], bx[NOP];
};

/* One step of a wave's rows: p <- the new field of the rows of c (c holds
 * NOP rows more on each side); SP: sponge, the pending factors spz, spx of
 * the previous field and nz, nx of the new one (row j's x factor in lane j). */
template <int NOP, int RX, bool VD, bool SP>
__device__ __forceinline__ void rows(const float (&c)[RX + 2 * NOP], float (&p)[RX + 2 * NOP], const float (&V)[RX],
                                     const float4 (&g)[VD ? RX : 1], const coef<NOP> &k, unsigned zmask, unsigned xint,
                                     float spz, float spx, float nz, float nx)
{
    /* no lane reads or masks hoisted out of the time loop */
    asm volatile("" : "+v"(spx), "+v"(nx), "+v"(xint));
    const int xi = __builtin_amdgcn_readfirstlane((int)xint);
#pragma unroll
    for (int j = 0; j < RX; j++) {
        const float cc = c[NOP + j];
        float zm[NOP], zp[NOP];
        zm[0] = up1(cc);
        zp[0] = dn1(cc);
#pragma unroll
        for (int i = 1; i < NOP; i++) {
            zm[i] = up1(zm[i - 1]);
            zp[i] = dn1(zp[i - 1]);
        }
        float pp = p[NOP + j];
        if (SP) {
            pp = pp * spz;
            pp = pp * row_factor(spx, j);
        }
        float lap = cc * k.c0;
#pragma unroll
        for (int i = 0; i < NOP; i++) {
            lap = lap + k.cz[i] * (zp[i] + zm[i]);
            lap = lap + k.cx[i] * (c[NOP + j + i + 1] + c[NOP + j - i - 1]);
        }
        if (VD) {
            float duz = 0.f, dux = 0.f;
#pragma unroll
            for (int i = 0; i < NOP; i++) {
                duz = duz + (zp[i] - zm[i]) * k.bz[i];
                dux = dux + (c[NOP + j + i + 1] - c[NOP + j - i - 1]) * k.bx[i];
            }
            const float4 gj = g[VD ? j : 0];
            const float dd = duz * gj.y + dux * gj.z;
            lap = lap - dd / gj.x;
        }
        const float t = 2.f * cc - pp;
        const float v = t + V[j] * lap;
        float nv = bits(zmask & (unsigned)__builtin_amdgcn_sbfe(xi, j, 1), v, pp);
        if (SP) {
            nv = nv * nz;
            nv = nv * row_factor(nx, j);
        }
        p[NOP + j] = nv;
        /* rows one after the other: interleaved, they take 3 times the
         * registers (no latency to hide between dependent VALU results) */
        __builtin_amdgcn_sched_barrier(0);
    }
}

/* two steps per exchange: 16 waves a block */
constexpr int nwave(int S) { return S == 2 ? AWEFD_RES_NWAVE2 : AWEFD_RES_NWAVE; }

template <int NOP, int RX, int S, bool VD>
__global__ __launch_bounds__(nwave(S) * WAVE) void k_cart2d_res(const awefd_res_args)
{
    constexpr int NW = nwave(S);
    using T = tile<NOP, RX, S, NW>;
    constexpr int NTHR = T::NTHR, H = T::H, EXT = T::EXT, ZW = T::ZW, OX = T::OX, ISH = T::ISH;
    extern __shared__ float img[];                     /* [2][rows + 2 NOP][64] */
    __shared__ int s_stop[2];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / WAVE);
    /* the arguments in constant memory (the kernel's own block) */
    const cargs &a = *(const cargs *)__builtin_amdgcn_kernarg_segment_ptr();
    const int lb = xcd_remap(blockIdx.x, a.ntz * a.ntx);
    const int tz = lb % a.ntz, txi = lb / a.ntz;
    const int n1 = a.n1, n2 = a.n2;
    const int z0 = tz * ZW - H, xb = txi * OX - H;     /* node of lane 0 and of image row 0 */
    const int iz = z0 + lane;
    const bool own = lane >= H && lane < WAVE - H && iz < n1;
    const bool zin = iz >= 0 && iz < n1;
    const int x0 = xb + NOP + wv * RX;                 /* first row of the wave */
    if (tid < 2) s_stop[tid] = 0;
    for (int i = tid; i < 2 * ISH; i += NTHR) img[i] = 0.f;

    /* per-node and per-row constants */
    const unsigned rowb = (unsigned)a.ld * 4u;
    const rsrc_t rV = mk_rsrc(a.vel, (unsigned)n2 * rowb);
    const rsrc_t rR = mk_rsrc(VD ? a.rho : a.vel, VD ? 4u * (unsigned)n2 * rowb : 0u);
    const unsigned vz = zin ? (unsigned)iz * 4u : OOB;
    const unsigned zmask = iz >= NOP && iz < n1 - NOP ? ~0u : 0u;
    const float spz = a.dabc && zin ? a.sp1[iz] : 1.f;
    /* the rows' x factors, row j in lane j */
    const float spx = a.dabc && lane < RX && x0 + lane >= 0 && x0 + lane < n2 ? a.sp2[x0 + lane] : 1.f;
    const bool sp = a.dabc && (z0 < a.nb || z0 + WAVE > n1 - a.nb || x0 < a.nb || x0 + RX > n2 - a.nb);
    float V[RX], A[RX + 2 * NOP], B[RX + 2 * NOP];
    float4 g[VD ? RX : 1];
    unsigned xint = 0;
#pragma unroll
    for (int j = 0; j < RX; j++) {
        const int ix = x0 + j;
        const bool in = ix >= 0 && ix < n2;
        V[j] = bld(rV, in ? vz : OOB, in ? (unsigned)ix * rowb : 0u);
        if (VD) {
            /* 0 beyond the grid: the quotient there is NaN, and masked */
            const unsigned vg = in && zin ? (unsigned)iz * 16u : OOB, sg = in ? 4u * (unsigned)ix * rowb : 0u;
            g[j] = make_float4(bld(rR, vg, sg), bld(rR, vg + 4u, sg), bld(rR, vg + 8u, sg), bld(rR, vg + 12u, sg));
        }
        xint |= ix >= NOP && ix < n2 - NOP ? 1u << j : 0u;
    }
    xint = __builtin_amdgcn_readfirstlane(xint);
#pragma unroll
    for (int j = 0; j < RX + 2 * NOP; j++) A[j] = B[j] = 0.f;
    coef<NOP> k;
    k.c0 = in_sgpr(a.c0);
#pragma unroll
    for (int i = 0; i < NOP; i++) {
        k.cz[i] = in_sgpr(a.cz[i]);
        k.cx[i] = in_sgpr(a.cx[i]);
        k.bz[i] = VD ? in_sgpr(a.bz[i]) : 0.f;
        k.bx[i] = VD ? in_sgpr(a.bx[i]) : 0.f;
    }

    const u64 *const E0 = a.E, *const E1 = a.E + (long)T::WORDS * a.ntz * a.ntx;   /* words by parity */
    const long me = (long)T::WORDS * (txi * a.ntz + tz);
    exchange<T, NOP> xch;
    xch.init(tid, tz, txi, a.ntz, a.ntx);
    const unsigned tag0 = a.tag0;

    /* source entries of this wave, one per lane (more than 64: re-read each
     * step); entries of one node are adjacent, rank counts those before */
    const int bucket = lb * NW + wv;
    const int ib = a.ibeg[bucket], ne = a.ibeg[bucket + 1] - ib;
    awefd_inj en = {0, 0, 0, 0, 0.f, 0.f, 0.f};
    if (lane < ne) en = a.inj[ib + lane];
    const int rank = node_rank(en, lane, ne < WAVE ? ne : WAVE);
    float amp = lane < ne ? a.wav[a.wexpl ? 0 : en.src] : 0.f;
    const float eV = lane < ne ? a.vel[(long)en.x * a.ld + en.z] : 0.f;
    /* a wave with sources stores its rows without the new field's sponge,
     * injects, then applies it */
    const float nspz = ne > 0 ? 1.f : spz, nspx = ne > 0 ? 1.f : spx;

    /* receivers of this block: the first of each thread in registers */
    const int nr = a.nr;
    const int rb = nr > 0 ? a.rbeg[lb] : 0, nrec = nr > 0 ? a.rbeg[lb + 1] - rb : 0;
    int r0 = -1, ro = 0;
    float rw[4] = {0.f, 0.f, 0.f, 0.f}, rsz[2] = {1.f, 1.f}, rsx[2] = {1.f, 1.f};
    if (tid < nrec) {
        r0 = a.ridx[rb + tid];
        const int jz = a.rj[3 * r0], jx = a.rj[3 * r0 + 1];
        ro = (jx - xb) * WAVE + jz - z0;
#pragma unroll
        for (int q = 0; q < 4; q++) rw[q] = a.rw[8 * r0 + q];
        if (a.dabc) {
            rsz[0] = a.sp1[jz];
            rsz[1] = a.sp1[jz + 1];
            rsx[0] = a.sp2[jx];
            rsx[1] = a.sp2[jx + 1];
        }
    }
    float *tr = a.tr + r0;                             /* this thread's trace, the next row's */
    __syncthreads();

    /* trace row it from the image of step it (the reference's u0: the
     * current field with its pending sponge factor; the factors are 1
     * without the sponge) */
    auto extract = [&](const float *I, int it) {
        if (r0 >= 0) {
            float s = 0.f;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                float u = I[ro + (q & 1) + (q >> 1) * WAVE];
                u = u * rsz[q & 1];
                u = u * rsx[q >> 1];
                const float t = u * rw[q];
                s = q == 0 ? t : s + t;
            }
            *tr = s;
            tr += nr;
        }
        if (__builtin_expect(nrec > NTHR, 0)) for (int i = tid + NTHR; i < nrec; i += NTHR) {
            const int r = a.ridx[rb + i], jz = a.rj[3 * r], jx = a.rj[3 * r + 1];
            const int o = (jx - xb) * WAVE + jz - z0;
            float s = 0.f;
            for (int q = 0; q < 4; q++) {
                float u = I[o + (q & 1) + (q >> 1) * WAVE];
                if (a.dabc) {
                    u = u * a.sp1[jz + (q & 1)];
                    u = u * a.sp2[jx + (q >> 1)];
                }
                const float t = u * a.rw[8 * r + q];
                s = q == 0 ? t : s + t;
            }
            a.tr[(long)it * nr + r] = s;
        }
    };

    /* one step: c <- the image of step it (own rows and NOP around them), p:
     * the previous field's rows, then the new ones, written to the other
     * image; PAR: the step's parity, XCH: it starts with an exchange */
    const int nt = a.nt;
    int dead = 0;
    auto step = [&]<int PAR, bool XCH>(int it, const u64 *words, float (&c)[RX + 2 * NOP], float (&p)[RX + 2 * NOP]) {
        float *const I = img + PAR * ISH, *const N = img + (PAR ^ 1) * ISH + (NOP + wv * RX) * WAVE;
        float na = 0.f;
        lds_barrier();
        if (XCH) {
            const unsigned tag = tag0 + (unsigned)it;
            xch.publish((u64 *)words + me, tag, I);
            xch.load(words);
            if (nrec > 0 && it > 0) extract(img + (PAR ^ 1) * ISH, it - 1);
            if (__builtin_expect(ne > 0, 0))
                if (lane < ne && it + 1 < nt) na = a.wav[(long)(it + 1) * a.wstride + (a.wexpl ? 0 : en.src)];
            if (__builtin_expect(!xch.finish(words, tag, I, a), 0)) s_stop[(it / S) & 1] = 1;
            lds_barrier();
        } else if (__builtin_expect(ne > 0, 0)) {
            if (lane < ne && it + 1 < nt) na = a.wav[(long)(it + 1) * a.wstride + (a.wexpl ? 0 : en.src)];
        }
        const float *Iw = I + wv * RX * WAVE + lane;
#pragma unroll
        for (int j = 0; j < RX + 2 * NOP; j++) c[j] = Iw[j * WAVE];
        if (XCH) dead = s_stop[(it / S) & 1];
        if (sp) rows<NOP, RX, VD, true>(c, p, V, g, k, zmask, xint, spz, spx, nspz, nspx);
        else rows<NOP, RX, VD, false>(c, p, V, g, k, zmask, xint, spz, spx, nspz, nspx);
        /* every computed node: with one step per exchange the margin comes
         * from the neighbours, with two a later step reads it */
        if (S > 1 || own) {
#pragma unroll
            for (int j = 0; j < RX; j++) N[j * WAVE + lane] = p[NOP + j];
        }
        if (__builtin_expect(ne > 0, 0)) {
            inject(a, en, rank, amp, eV, ib, ne, lane, it, N, x0, z0);
            if (sp)
                for (int r = 0; r < RX; r++) {
                    const int x = x0 + r;
                    if (x < 0 || x >= n2) continue;
                    float w = N[r * WAVE + lane];
                    w = w * spz;
                    w = w * a.sp2[x];
                    N[r * WAVE + lane] = w;
                }
            amp = na;
        }
        /* the gradient keeps every field: the owned nodes (the next poll's
         * wait covers the stores) */
        if (__builtin_expect(a.F != nullptr, 0) && it + 1 < nt) {
            const rsrc_t rF = mk_rsrc(a.F + (long)it * a.nal, (unsigned)n2 * rowb);
#pragma unroll
            for (int j = 0; j < RX; j++) {
                const int lr = wv * RX + j;
                const bool in = lr >= EXT && lr < EXT + OX && x0 + j < n2;
                bst<2>(rF, in && own ? (unsigned)iz * 4u : OOB, in ? (unsigned)(x0 + j) * rowb : 0u,
                       ne > 0 ? N[j * WAVE + lane] : p[NOP + j]);
            }
        }
        /* between exchanges the image of this step is overwritten next */
        if (S > 1 && XCH && nrec > 0) extract(I, it);
        if (XCH) dead = __builtin_amdgcn_readfirstlane(dead);
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
    /* a block that gave up tells the others and the host */
    if (dead) {
        if (tid == 0) __hip_atomic_store(a.stop, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        return;
    }
    if (S == 1 || !(nt & 1)) {
        lds_barrier();
        extract(img + ((nt - 1) & 1) * ISH, nt - 1);
    }
    /* the last two fields: the newest from the image, the one before from
     * the rows it was computed from */
    const rsrc_t rC = mk_rsrc(a.C, (unsigned)n2 * rowb), rP = mk_rsrc(a.P, (unsigned)n2 * rowb);
    const float *Iw = img + (nt & 1) * ISH + (NOP + wv * RX) * WAVE + lane;
    if (nt & 1) {
#pragma unroll
        for (int j = 0; j < RX; j++) B[NOP + j] = A[NOP + j];
    }
    const unsigned vzo = own ? (unsigned)iz * 4u : OOB;
#pragma unroll
    for (int j = 0; j < RX; j++) {
        const int lr = wv * RX + j;                    /* row of the computed ones */
        const bool in = lr >= EXT && lr < EXT + OX && x0 + j < n2;
        const unsigned s = in ? (unsigned)(x0 + j) * rowb : 0u, v = in ? vzo : OOB;
        bst(rC, v, s, Iw[j * WAVE]);
        bst(rP, v, s, B[NOP + j]);
    }
}

template <int NOP, int RX, int S, bool VD>
struct kernel {
    static constexpr size_t LDS = sizeof(float) * 2 * (size_t)tile<NOP, RX, S, nwave(S)>::ISH;
    static constexpr int NTHR = nwave(S) * WAVE;

    static hipError_t attr()
    {
        if (LDS <= 65536) return hipSuccess;
        return hipFuncSetAttribute((const void *)k_cart2d_res<NOP, RX, S, VD>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS);
    }
    static int launch(const awefd_res_args *one, int nblk, hipStream_t s)
    {
        const hipError_t e = attr();
        if (e != hipSuccess) return (int)e;
        awefd_res_args a = *one;
        void *args[] = {&a};
        return (int)hipLaunchCooperativeKernel((const void *)k_cart2d_res<NOP, RX, S, VD>, dim3(nblk), dim3(NTHR), args,
                                               (unsigned)LDS, s);
    }
    static int blocks()
    {
        int nb = 0;
        if (attr() != hipSuccess) return 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, (const void *)k_cart2d_res<NOP, RX, S, VD>, NTHR, LDS) !=
            hipSuccess)
            return 0;
        return nb;
    }
};

/* f<kernel> for a compiled tile (awefd_res_rows) */
template <int NOP, class F>
int pick(int rx, int S, int vd, F f)
{
#define RX_CASE(n, s, v) case n: return f(kernel<NOP, n, s, v>());
    if (S == 2 && vd) switch (rx) {
        RX_CASE(1, 2, true) RX_CASE(2, 2, true) RX_CASE(3, 2, true) RX_CASE(4, 2, true)
    }
    if (S == 2 && !vd) switch (rx) {
        RX_CASE(1, 2, false) RX_CASE(2, 2, false) RX_CASE(3, 2, false) RX_CASE(4, 2, false) RX_CASE(5, 2, false)
        RX_CASE(6, 2, false)
    }
    if (S == 1 && !vd) switch (rx) {
        RX_CASE(8, 1, false) RX_CASE(10, 1, false) RX_CASE(12, 1, false) RX_CASE(14, 1, false) RX_CASE(16, 1, false)
        RX_CASE(18, 1, false) RX_CASE(20, 1, false) RX_CASE(22, 1, false) RX_CASE(24, 1, false) RX_CASE(26, 1, false)
        RX_CASE(28, 1, false) RX_CASE(30, 1, false) RX_CASE(32, 1, false)
    }
#undef RX_CASE
    return -1;
}

} // namespace

#define RES_CAT2(a, b) a##b
#define RES_CAT(a, b) RES_CAT2(a, b)

extern "C" int RES_CAT(awefd__res_launch, RES_NOP)(const awefd_res_args *a, int nblk, int rx, int S, int vd, void *stream)
{
    const int e = pick<RES_NOP>(rx, S, vd, [&](auto k) { return k.launch(a, nblk, (hipStream_t)stream); });
    return e < 0 ? (int)hipErrorInvalidValue : e;
}

extern "C" int RES_CAT(awefd__res_blocks, RES_NOP)(int rx, int S, int vd)
{
    const int n = pick<RES_NOP>(rx, S, vd, [&](auto k) { return k.blocks(); });
    return n > 0 ? n : 0;
}
