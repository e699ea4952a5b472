/*
 * Resident adjoint of the cartesian 2-D loop for gfx950 (MI355X): every
 * backward step of a shot whose forward fields are all stored, in one
 * cooperative launch.  Tiles, rim exchange and its protocol are res_loop.h's,
 * one step per exchange.
 *
 * A backward step of a 400 x 800 shot is 28 bytes a node, 9 MB, from the
 * Infinity Cache, but as a launch it took 7.6 us, most of it the latency of
 * its loads.  Here alpha_{n+1}, alpha_{n+2}, V and dJ/dV stay in registers,
 * y = V M G alpha_{n+1} in LDS, whose rim is all the neighbours need, and only
 * c_n is read, a step ahead: 2.9 us a step.  Up to 12 rows a wave fit the
 * registers with fdorder 2 and 4 (1.5 M padded nodes at best), 10 with 6
 * (1.2 M) and 8 with 8 (0.9 M); larger grids keep a launch per step.
 *
 * Arithmetic, order and selections are adj_body's (adj_kernels.hip) node for
 * node: the same bits.
 */
#include "res_adj.h"
#include "res_tile.h"

#pragma clang fp contract(off)

namespace {

template <int NOP, int RX>
__global__ __launch_bounds__(AWEFD_RES_NWAVE * WAVE) void k_adj_res(const awefd_resadj_args a)
{
    using T = tile<NOP, RX, 1>;
    constexpr int NTHR = T::NTHR, H = T::H, ZW = T::ZW, OX = T::OX, ISH = T::ISH, R = RX + 2 * NOP;
    extern __shared__ float img[];                     /* [2][rows + 2 NOP][64] */
    __shared__ int s_stop[2];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int lb = xcd_remap(blockIdx.x, a.ntz * a.ntx);
    const int tz = lb % a.ntz, txi = lb / a.ntz;
    const int nz = a.nz, nx = a.nx;
    const int z0 = tz * ZW - H, x0 = txi * OX + wv * RX;   /* node of lane 0, first row of the wave */
    const int iz = z0 + lane;
    const bool own = lane >= H && lane < WAVE - H && iz < nz;
    const bool zin = iz >= 0 && iz < nz;
    if (tid < 2) s_stop[tid] = 0;
    for (int i = tid; i < 2 * ISH; i += NTHR) img[i] = 0.f;

    const unsigned rowb = (unsigned)a.ld * 4u, nbytes = (unsigned)nx * rowb;
    const rsrc_t rV = mk_rsrc(a.V, nbytes);
    const unsigned vz = zin ? (unsigned)iz * 4u : OOB;
    const unsigned zmask = iz >= NOP && iz < nz - NOP ? ~0u : 0u;
    const float gz = a.sp1[min(max(iz, 0), nz - 1)];
    /* the rows' x factors, row j in lane j */
    const float gx = a.sp2[min(x0 + lane, nx - 1)];
    float V[RX], G[RX], A[RX], B[RX], c[R], d[R];
    unsigned xint = 0;
#pragma unroll
    for (int j = 0; j < RX; j++) {
        const int ix = x0 + j;
        V[j] = bld(rV, ix < nx ? vz : OOB, ix < nx ? (unsigned)ix * rowb : 0u);
        xint |= ix >= NOP && ix < nx - NOP ? 1u << j : 0u;
        A[j] = B[j] = G[j] = 0.f;
    }
    /* rows x0 - NOP .. of c_n */
    auto fields = [&](float (&q)[R], int n) {
        const rsrc_t rC = mk_rsrc(n == 0 ? a.c0f : a.seg + (long)(n - 1) * a.nal, nbytes);
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int ix = x0 - NOP + r;
            const bool in = ix >= 0 && ix < nx;
            q[r] = bld<2>(rC, in ? vz : OOB, in ? (unsigned)ix * rowb : 0u);
        }
    };
    const int nt = a.nt;
    fields(c, nt - 1);

    const float k0 = in_sgpr(a.c0);
    float kz[NOP], kx[NOP];
#pragma unroll
    for (int k = 0; k < NOP; k++) {
        kz[k] = in_sgpr(a.cz[k]);
        kx[k] = in_sgpr(a.cx[k]);
    }

    const u64 *const E0 = a.E, *const E1 = a.E + (long)T::WORDS * a.ntz * a.ntx;   /* words by parity */
    const long me = (long)T::WORDS * (txi * a.ntz + tz);
    exchange<T, NOP> xch;
    xch.init(tid, tz, txi, a.ntz, a.ntx);
    const unsigned tag0 = a.tag0;

    /* receiver and source entries of this wave's rows, the first 64 one per
     * lane with their amplitudes of the coming step */
    const int col = tz + a.ntz * (txi * AWEFD_RES_NWAVE + wv);
    const int rb = a.rbeg[col], rn = a.rbeg[col + 1] - rb, sb = a.sbeg[col], sn = a.sbeg[col + 1] - sb;
    int rz = 0, rx = 0, rs = 0, sz = 0, sx = 0, ss = 0;
    float rw = 0.f, sw = 0.f;
    if (lane < rn) {
        const awefd_inj &e = a.rinj[rb + lane];
        rz = e.z;
        rx = e.x;
        rs = e.src;
        rw = e.w;
    }
    if (lane < sn) {
        const awefd_inj &e = a.sinj[sb + lane];
        sz = e.z;
        sx = e.x;
        ss = e.src;
        sw = e.w;
    }
    auto residual = [&](int src, int n) { return a.res[(long)n * a.nr + src]; };
    auto wavelet = [&](int src, int n) { return a.wav[(long)n * a.wstride + src]; };
    float ramp = lane < rn ? residual(rs, nt - 1) : 0.f, samp = lane < sn ? wavelet(ss, nt - 1) : 0.f;
    __syncthreads();

    int dead = 0;
    /* backward step n (the i-th): a1 alpha_{n+1}, a2 alpha_{n+2}, then
     * alpha_n; q c_n, next c_{n-1} */
    auto step = [&]<int PAR>(int i, const u64 *words, float (&a1)[RX], float (&a2)[RX], float (&q)[R],
                             float (&next)[R]) {
        float *const I = img + PAR * ISH, *const N = img + (PAR ^ 1) * ISH + (NOP + wv * RX) * WAVE + lane;
        const int n = nt - 1 - i;
        const unsigned tag = tag0 + (unsigned)i;
        lds_barrier();
        xch.publish((u64 *)words + me, tag, I);
        xch.load(words);
        if (__builtin_expect(!xch.finish(words, tag, I, a), 0)) s_stop[i & 1] = 1;
        lds_barrier();
        float y[R], nr = 0.f, ns = 0.f;
        const float *Iw = I + wv * RX * WAVE + lane;
#pragma unroll
        for (int r = 0; r < R; r++) y[r] = Iw[r * WAVE];
        dead = s_stop[i & 1];
        if (n > 0) {
            fields(next, n - 1);
            if (lane < rn) nr = residual(rs, n - 1);
            if (lane < sn) ns = wavelet(ss, n - 1);
        }
        float t[RX], g[RX], gv[RX];
        float fx = gx;
        asm volatile("" : "+v"(fx));                   /* no lane reads hoisted out of the loop */
#pragma unroll
        for (int j = 0; j < RX; j++) {
            const int r = NOP + j;
            const unsigned in = zmask & ((xint >> j) & 1u ? ~0u : 0u);
            g[j] = gz * row_factor(fx, j);
            t[j] = g[j] * a1[j];
            float zm = y[r], zp = y[r], ly = k0 * y[r];
#pragma unroll
            for (int k = 1; k <= NOP; k++) {
                zm = up1(zm);
                zp = dn1(zp);
                ly = ly + kz[k - 1] * (zp + zm) + kx[k - 1] * (y[r + k] + y[r - k]);
            }
            zm = zp = q[r];
            float lc = k0 * q[r];
#pragma unroll
            for (int k = 1; k <= NOP; k++) {
                zm = up1(zm);
                zp = dn1(zp);
                lc = lc + kz[k - 1] * (zp + zm) + kx[k - 1] * (q[r + k] + q[r - k]);
            }
            const float tb = g[j] * a2[j];
            a2[j] = bits(in, 2.f * t[j], 0.f) + ly + g[j] * bits(in, -tb, tb);
            gv[j] = bits(in, lc * t[j], 0.f);
        }
        auto receive = [&](int qz, int qx, float qa) {
#pragma unroll
            for (int j = 0; j < RX; j++) a2[j] = (qz == iz && qx == x0 + j) ? a2[j] + g[j] * qa : a2[j];
        };
        auto inject = [&](int qz, int qx, float qa) {
#pragma unroll
            for (int j = 0; j < RX; j++) gv[j] = (qz == iz && qx == x0 + j) ? gv[j] + qa * t[j] : gv[j];
        };
        const float rv = ramp * rw, sv = samp * sw;
        for (int l = 0; l < min(rn, WAVE); l++)
            receive(__builtin_amdgcn_readlane(rz, l), __builtin_amdgcn_readlane(rx, l), row_factor(rv, l));
        for (int e = WAVE; e < rn; e++)
            receive(a.rinj[rb + e].z, a.rinj[rb + e].x, residual(a.rinj[rb + e].src, n) * a.rinj[rb + e].w);
        for (int l = 0; l < min(sn, WAVE); l++)
            inject(__builtin_amdgcn_readlane(sz, l), __builtin_amdgcn_readlane(sx, l), row_factor(sv, l));
        for (int e = WAVE; e < sn; e++)
            inject(a.sinj[sb + e].z, a.sinj[sb + e].x, wavelet(a.sinj[sb + e].src, n) * a.sinj[sb + e].w);
        ramp = nr;
        samp = ns;
#pragma unroll
        for (int j = 0; j < RX; j++) {
            G[j] = G[j] + gv[j];
            const unsigned in = zmask & ((xint >> j) & 1u ? ~0u : 0u);
            if (own) N[j * WAVE] = bits(in, V[j] * (g[j] * a2[j]), 0.f);
        }
        dead = __builtin_amdgcn_readfirstlane(dead);
    };

    for (int i = 0; i < nt; i += 2) {
        step.template operator()<0>(i, E0, A, B, c, d);
        if (__builtin_expect(dead, 0) || i + 1 >= nt) break;
        step.template operator()<1>(i + 1, E1, B, A, d, c);
        if (__builtin_expect(dead, 0)) break;
    }
    /* a block that gave up tells the others and the host */
    if (dead) {
        if (tid == 0) __hip_atomic_store(a.stop, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        return;
    }
    const rsrc_t rG = mk_rsrc(a.gV, nbytes);
#pragma unroll
    for (int j = 0; j < RX; j++)
        bst(rG, own && x0 + j < nx ? vz : OOB, x0 + j < nx ? (unsigned)(x0 + j) * rowb : 0u, G[j]);
}

template <int NOP, int RX>
struct kernel {
    static constexpr int NTHR = AWEFD_RES_NWAVE * WAVE;
    static constexpr size_t LDS = sizeof(float) * 2 * (size_t)tile<NOP, RX, 1>::ISH;

    static hipError_t attr()
    {
        if (LDS <= 65536) return hipSuccess;
        return hipFuncSetAttribute((const void *)k_adj_res<NOP, RX>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS);
    }
    static int launch(const awefd_resadj_args *one, int nblk, hipStream_t s)
    {
        const hipError_t e = attr();
        if (e != hipSuccess) return (int)e;
        awefd_resadj_args a = *one;
        void *args[] = {&a};
        return (int)hipLaunchCooperativeKernel((const void *)k_adj_res<NOP, RX>, dim3(nblk), dim3(NTHR), args,
                                               (unsigned)LDS, s);
    }
    static int blocks()
    {
        int nb = 0;
        if (attr() != hipSuccess) return 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, (const void *)k_adj_res<NOP, RX>, NTHR, LDS) != hipSuccess)
            return 0;
        return nb;
    }
};

/* f<kernel> for a compiled tile (resadj_pick's list), without those that
 * would spill (about 19 VGPRs a row and 28 a stencil node) */
template <int NOP, class F>
int pick_rx(int rx, F f)
{
    switch (rx) {
#define RX_CASE(n) \
    case n: \
        if constexpr (19 * n + 28 * NOP <= 290) return f(kernel<NOP, n>()); \
        break;
    RX_CASE(1) RX_CASE(2) RX_CASE(3) RX_CASE(4) RX_CASE(5) RX_CASE(6) RX_CASE(8) RX_CASE(10) RX_CASE(12)
#undef RX_CASE
    }
    return -1;
}

template <class F>
int pick(int nop, int rx, F f)
{
    switch (nop) {
    case 1: return pick_rx<1>(rx, f);
    case 2: return pick_rx<2>(rx, f);
    case 3: return pick_rx<3>(rx, f);
    case 4: return pick_rx<4>(rx, f);
    }
    return -1;
}

} // namespace

extern "C" int awefd__resadj_launch(const awefd_resadj_args *a, int nblk, int nop, int rx, void *stream)
{
    const int e = pick(nop, rx, [&](auto k) { return k.launch(a, nblk, (hipStream_t)stream); });
    return e < 0 ? (int)hipErrorInvalidValue : e;
}

extern "C" int awefd__resadj_blocks(int nop, int rx)
{
    const int n = pick(nop, rx, [&](auto k) { return k.blocks(); });
    return n > 0 ? n : 0;
}
