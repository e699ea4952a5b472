/* Resident 2-D loop, stencil half-width 4 (fdorder 8). */
#define RES_NOP 4
#include "res_loop.h"
