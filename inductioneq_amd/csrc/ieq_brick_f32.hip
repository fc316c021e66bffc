#define IEQ_BRICK_REAL float
#include "ieq_brick.inc"
