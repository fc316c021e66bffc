#define IEQ_BRICK_REAL double
#include "ieq_brick.inc"
