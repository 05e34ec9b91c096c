// exl3_rate_gemm.hip -- one rate's instantiation of the EXL3 GEMM kernels,
// compiled once per K (0..8) with -DEXL3_INST_K=K like exl3_rate.hip: K =
// 1..8 the integer rates, K = 0 the half-integer rates n = 24, 40.
#include "exl3_kern.h"

#ifndef EXL3_INST_K
#error "exl3_rate_gemm.hip is built with -DEXL3_INST_K=<rate>"
#endif

namespace exl3 {

#if EXL3_INST_K > 0
template EXL3_GEMM_GO(EXL3_INST_K);
template EXL3_GEMM_GROUPED_GO(EXL3_INST_K);
template EXL3_GEMM_RD_GROUPED_GO(EXL3_INST_K);
template EXL3_GEMM_RD_GO(EXL3_INST_K, 0);
#else
template EXL3_GEMM_FRAC_GO(3);
template EXL3_GEMM_FRAC_GO(5);
template EXL3_GEMM_RD_GO(1, 3);
template EXL3_GEMM_RD_GO(1, 5);
#endif

}  // namespace exl3
