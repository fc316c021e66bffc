#define IEQ_NODE_REAL double
#include "ieq_node_stage.inc"
