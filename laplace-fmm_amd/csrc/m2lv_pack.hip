// m2lv_pack.hip -- class-major packing of a level's multipoles for the FP64
// vector M2L (m2lv.h).
#include "device_common.h"
#include "m2lv.h"

namespace lfmm {

// A wave handles 16 parents x 4 consecutive coefficients (per class): it reads
// 64 bytes of each child and writes 256 consecutive bytes per coefficient.
__global__ void __launch_bounds__(256) k_m2lv_pack(const double2* __restrict__ src, int64_t stride, int nx, int parents,
                                                  const int32_t* __restrict__ child_begin,
                                                  const uint64_t* __restrict__ child_keys, int slots,
                                                  double2* __restrict__ out)
{
    const int p = xcd_local_block(blockIdx.x, gridDim.x) * 16 + (threadIdx.x & 15);
    if (p >= slots) return;
    int box[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) box[s] = -1;
    if (p < parents) {
        const int b = child_begin[p], e = child_begin[p + 1];
        uint32_t present = 0;
        for (int i = b; i < e; ++i) present |= 1u << (int)(child_keys[i] & 7u);
#pragma unroll
        for (int s = 0; s < 8; ++s)
            if ((present >> s) & 1u) box[s] = b + __popc(present & ((1u << s) - 1u));
    }
    for (int k = threadIdx.x >> 4; k < nx; k += 16) {
        double2 v[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) v[s] = box[s] < 0 ? make_double2(0.0, 0.0) : src[(int64_t)box[s] * stride + k];
#pragma unroll
        for (int s = 0; s < 8; ++s) out[((int64_t)s * nx + k) * slots + p] = v[s];
    }
}

hipError_t launch_m2lv_pack(const RtrLevel& L, int nx, double2* packed, hipStream_t st)
{
    // every parent of the level, also when the targets are a list of them
    const int slots = m2lv_slots(L.num_parents);
    hipLaunchKernelGGL(k_m2lv_pack, dim3((unsigned)((slots + 15) / 16)), dim3(256), 0, st, L.src,
                       (int64_t)(L.stride > 0 ? L.stride : nx), nx, L.num_parents, L.child_begin, L.child_keys, slots,
                       packed);
    return hipGetLastError();
}

}  // namespace lfmm
