#define IEQ_NODE_REAL float
#include "ieq_node_stage.inc"
