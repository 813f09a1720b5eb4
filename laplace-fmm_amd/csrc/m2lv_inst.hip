// m2lv_inst.hip -- instantiates the FP64 vector M2L, M2M and L2L for one expansion size
// (LFMM_N, set by the build).
#include "m2lv_kernels.h"

#ifndef LFMM_N
#error "build with -DLFMM_N=<terms>"
#endif

namespace lfmm {
template hipError_t do_m2lv<LFMM_N>(int, const M2LStepTables&, const M2lvTables&, const M64Level&, hipStream_t);
}  // namespace lfmm
