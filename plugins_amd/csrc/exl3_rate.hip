// exl3_rate.hip -- one rate's instantiation of the EXL3 GEMV and grouped MoE
// GEMV kernels.  The build compiles this file once per K with -DEXL3_INST_K=K:
// K = 1..8 are the integer rates n = 16K with compile-time bit windows, K = -3
// and -5 the half-integer rates n = 24 and 40, K = 0 the run-time window form
// for any even n.
#include "exl3_kern.h"

#ifndef EXL3_INST_K
#error "exl3_rate.hip is built with -DEXL3_INST_K=<rate>"
#endif

namespace exl3 {

template EXL3_GEMV_GO(EXL3_INST_K);
template EXL3_MOE_GEMV_GO(EXL3_INST_K);

}  // namespace exl3
