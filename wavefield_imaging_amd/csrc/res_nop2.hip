/* Resident 2-D loop, stencil half-width 2 (fdorder 4). */
#define RES_NOP 2
#include "res_loop.h"
