/* Resident 2-D loop, stencil half-width 3 (fdorder 6). */
#define RES_NOP 3
#include "res_loop.h"
