// m2l64_inst.hip -- instantiates the FP64 matrix-core M2L for one expansion
// size (LFMM_N, set by the build).
#include "m2l64_kernels.h"

#ifndef LFMM_N
#error "build with -DLFMM_N=<terms>"
#endif

namespace lfmm {
template hipError_t do_m2l64<LFMM_N>(const M2LStepTables&, const M64Tables&, const M64Level&, hipStream_t);
}  // namespace lfmm
