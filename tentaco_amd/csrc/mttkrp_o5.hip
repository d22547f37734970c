// Order-5 MTTKRP kernels.
#include "mttkrp_order.h"

TT_INSTANTIATE_ORDER(5)
