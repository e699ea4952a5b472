/*
 * Tile, rim exchange and lane helpers of the resident 2-D loops (res_loop.h,
 * res_polar.hip): see res_loop.h for the protocol and its measurements.
 */
#ifndef AWEFD_RES_TILE_H
#define AWEFD_RES_TILE_H
#include <hip/hip_runtime.h>
#include "awefd_hip.h"
#include "awefd_internal.h"

#pragma clang fp contract(off)

namespace {

using namespace awefd;

typedef unsigned long long u64;
__device__ __forceinline__ void put_word(u64 *p, unsigned tag, float v)
{
    __hip_atomic_store(p, ((u64)tag << 32) | __builtin_bit_cast(unsigned, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 get_word(const u64 *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ float row_factor(float v, int j)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), j));
}

/* lane i receives lane i-1 / i+1; the lane without a source gets 0 */
__device__ __forceinline__ float up1(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float dn1(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x130, 0xf, 0xf, true));
}

/* The tile and its margin; NW: waves of its block. */
template <int NOP, int RX, int S, int NW = AWEFD_RES_NWAVE>
struct tile {
    static constexpr int NTHR = NW * WAVE;
    static constexpr int H = S * NOP;                  /* margin of the image   */
    static constexpr int EXT = (S - 1) * NOP;          /* ... that is computed  */
    static constexpr int ZW = WAVE - 2 * H;            /* owned z lanes         */
    static constexpr int TX = NW * RX;                 /* computed rows         */
    static constexpr int OX = TX - 2 * EXT;            /* owned rows            */
    static constexpr int ROWS = TX + 2 * NOP;          /* image rows            */
    static constexpr int ISH = ROWS * WAVE;            /* floats of one image   */
    static_assert(ZW > 0 && OX >= H, "tile too small for its margin");
    /* words of the rim: low-z nodes [row][H], high-z nodes [row][H], the
     * first H rows, the last H rows (64 words each, the owned lanes' used),
     * each part on lines of its own (16 words) */
    static constexpr int NZ = OX * H, NX = H * ZW;
    static constexpr int ZH = (NZ + 15) / 16 * 16, XL = 2 * ZH, XH = XL + H * WAVE, WORDS = XH + H * WAVE;
    /* words polled: the neighbours' opposite sides and a K x K corner of the
     * diagonal ones (the trace extraction reads 1; two steps read H) */
    static constexpr int K = S == 1 ? 1 : H;
    static constexpr int HALO = 2 * NZ + 2 * NX + 4 * K * K;
    static constexpr int MW = (HALO + NTHR - 1) / NTHR, MP = (WORDS + NTHR - 1) / NTHR;
};

constexpr unsigned NONE = 0xffffffffu;

/* One thread's share of the exchange: up to MP words it publishes (image
 * node, byte offset in the block's words) and MW words it polls (byte offset
 * in the parity's words, image node). */
template <class T, int NOP>
struct exchange {
    static constexpr int MW = T::MW, MP = T::MP;
    unsigned psrc[MP], pout[MP];
    unsigned src[MW];
    int dst[MW];
    u64 v[MW];

    __device__ __forceinline__ void init(int tid, int tz, int txi, int ntz, int ntx)
    {
        constexpr int H = T::H, ZW = T::ZW, K = T::K, W = T::WORDS;
#pragma unroll
        for (int i = 0; i < MP; i++) {
            const int w = tid + i * T::NTHR;
            int at = -1;
            if (w < T::NZ) at = (H + w / H) * WAVE + H + w % H;
            else if (w >= T::ZH && w < T::ZH + T::NZ) at = (H + (w - T::ZH) / H) * WAVE + WAVE - 2 * H + (w - T::ZH) % H;
            else if (w >= T::XL && w < T::XH) at = H * WAVE + w - T::XL;
            else if (w >= T::XH && w < W) at = T::OX * WAVE + w - T::XH;
            psrc[i] = at < 0 ? 0u : (unsigned)at;
            pout[i] = at < 0 ? NONE : 8u * (unsigned)w;
        }
        const int b = txi * ntz + tz;
        const bool lz = tz > 0, hz = tz + 1 < ntz, lx = txi > 0, hx = txi + 1 < ntx;
#pragma unroll
        for (int i = 0; i < MW; i++) {
            int w = tid + i * T::NTHR, s = -1;
            dst[i] = 0;
            if (w < T::NZ) {                           /* z below: lanes 0..H-1 */
                if (lz) s = (b - 1) * W + T::ZH + w;
                dst[i] = (H + w / H) * WAVE + w % H;
            } else if ((w -= T::NZ) < T::NZ) {         /* z above: the last H lanes */
                if (hz) s = (b + 1) * W + w;
                dst[i] = (H + w / H) * WAVE + WAVE - H + w % H;
            } else if ((w -= T::NZ) < T::NX) {         /* x below: image rows 0..H-1 */
                const int at = w / ZW * WAVE + H + w % ZW;
                if (lx) s = (b - ntz) * W + T::XH + at;
                dst[i] = at;
            } else if ((w -= T::NX) < T::NX) {         /* x above: rows after the owned */
                const int at = w / ZW * WAVE + H + w % ZW;
                if (hx) s = (b + ntz) * W + T::XL + at;
                dst[i] = (H + T::OX) * WAVE + at;
            } else if ((w -= T::NX) < 4 * K * K) {     /* corners of the diagonal blocks */
                const int q = w / (K * K), h = w % (K * K) / K, k = w % K;
                const int zu = q & 1, xu = q >> 1;     /* above in z, in x */
                if ((zu ? hz : lz) && (xu ? hx : lx))
                    s = (b + (zu ? 1 : -1) + (xu ? ntz : -ntz)) * W + (xu ? T::XL + h * WAVE : T::XH + (H - K + h) * WAVE)
                        + (zu ? H + k : WAVE - H - K + k);
                dst[i] = (xu ? H + T::OX + h : H - K + h) * WAVE + (zu ? WAVE - H + k : H - K + k);
            }
            src[i] = s < 0 ? NONE : (unsigned)s * 8u;
        }
    }

    __device__ __forceinline__ void publish(u64 *mine, unsigned tag, const float *img)
    {
#pragma unroll
        for (int i = 0; i < MP; i++)
            if (pout[i] != NONE) put_word((u64 *)((char *)mine + pout[i]), tag, img[psrc[i]]);
    }

    __device__ __forceinline__ void load(const u64 *words)
    {
#pragma unroll
        for (int i = 0; i < MW; i++)
            if (src[i] != NONE) v[i] = get_word((const u64 *)((const char *)words + src[i]));
    }

    /* with the words of load(): wait for those of `tag`, put them into the
     * image; false: given up */
    template <class A>
    __device__ __forceinline__ bool finish(const u64 *words, unsigned tag, float *img, const A &a)
    {
        unsigned tries = 0;
        long long t0 = 0;
        for (;;) {
            bool bad = false;
#pragma unroll
            for (int i = 0; i < MW; i++) bad |= src[i] != NONE && (unsigned)(v[i] >> 32) != tag;
            if (!__any(bad)) break;
            load(words);
            if (__builtin_expect((++tries & a.wmask) == 0, 0)) {
                const long long now = wall_clock64();
                if (t0 == 0) t0 = now;
                if (now - t0 > a.wticks ||
                    __hip_atomic_load(a.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != 0u)
                    return false;
            }
        }
#pragma unroll
        for (int i = 0; i < MW; i++)
            if (src[i] != NONE) img[dst[i]] = __builtin_bit_cast(float, (unsigned)v[i]);
        return true;
    }
};

/* A barrier that orders the block's LDS accesses only: __syncthreads would
 * also wait for the acknowledgements of the rim words and traces just
 * stored (0.4 us of a step). */
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

/* The value stays in a scalar register: its load is not repeated where it is
 * used. */
__device__ __forceinline__ float in_sgpr(float v)
{
    asm volatile("" : "+s"(v));
    return v;
}

/* m's bits from a, the others from b (one v_bfi_b32: a select the compiler
 * does not turn into a branch around the stencil) */
__device__ __forceinline__ float bits(unsigned m, float a, float b)
{
    return __builtin_bit_cast(float, (m & __builtin_bit_cast(unsigned, a)) | (~m & __builtin_bit_cast(unsigned, b)));
}

} // namespace

#endif
