// Order-4 MTTKRP kernels.
#include "mttkrp_order.h"

TT_INSTANTIATE_ORDER(4)
