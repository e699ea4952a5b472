/*
 * Arguments and launcher of the resident adjoint loop (res_adj.hip).
 */
#ifndef AWEFD_RES_ADJ_H
#define AWEFD_RES_ADJ_H
#include "awefd_internal.h"

#ifdef __cplusplus
extern "C" {
#endif

typedef struct {
    int nz, nx, ld;              /* padded grid, row stride                    */
    int ntz, ntx;                /* tiles                                      */
    int nt;
    const float *c0f, *seg;      /* c_0, and c_n at seg + (n - 1) nal          */
    long nal;
    const float *V;              /* (v dt)^2                                   */
    float *gV;                   /* dJ/dV (padded grid), written               */
    const float *sp1, *sp2;      /* sponge factors per axis (ones without)     */
    float c0, cz[AWEFD_RES_MAXNOP], cx[AWEFD_RES_MAXNOP];
    /* receiver and source nodes per wave: bucket tz + ntz (8 tx + wave) */
    const int *rbeg, *sbeg;
    const awefd_inj *rinj, *sinj;
    const float *res;            /* residual rows (nt x nr)                    */
    int nr;
    const float *wav;
    long wstride;
    unsigned long long *E;       /* rim words, as awefd_res_args'              */
    unsigned tag0;
    unsigned *stop;
    unsigned wmask;
    long long wticks;
} awefd_resadj_args;

/* every backward step of one grid, cooperative; resident blocks per CU (0:
 * not compiled) */
int awefd__resadj_launch(const awefd_resadj_args *a, int nblk, int nop, int rx, void *stream);
int awefd__resadj_blocks(int nop, int rx);

#ifdef __cplusplus
}
#endif

#endif
