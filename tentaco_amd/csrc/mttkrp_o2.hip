// Order-2 MTTKRP kernels.
#include "mttkrp_order.h"

TT_INSTANTIATE_ORDER(2)
