/* Resident 2-D loop, stencil half-width 1 (fdorder 2). */
#define RES_NOP 1
#include "res_loop.h"
