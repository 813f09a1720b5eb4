// rowbc.h -- FP64 products with a coefficient broadcast from a register that
// holds 16 of them, one per lane of each 16-lane row (row_newbcast, full rate;
// the compiler does not fold the broadcast into the product).  The coefficient
// register is to be written by a load: less than 2 wait states after a vector
// instruction wrote it the broadcast would read the old value, and the compiler,
// which cannot see into the assembly, may copy or reload a spilled register there.
// check_dpp.py looks for that in every built library.
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>

namespace lfmm {

template <int B, int E, typename F>
__device__ __forceinline__ void sfor2(F&& f)
{
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        sfor2<B + 1, E>(f);
    }
}

// acc += (entry I of c's 16-lane row) * x
template <int I>
__device__ __forceinline__ void fmac_bc(double& acc, double c, double x)
{
    asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(c), "v"(x), "n"(I));
}
// acc -= (entry I of c's 16-lane row) * x
template <int I>
__device__ __forceinline__ void fnmac_bc(double& acc, double c, double x)
{
    asm("v_fmac_f64_dpp %0, %1, -%2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(c), "v"(x), "n"(I));
}
// entry I of c's 16-lane row in every lane
template <int I>
__device__ __forceinline__ double bc(double c)
{
    double r;
    asm("v_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(c), "n"(I));
    return r;
}

#define LFMM_BC(I) " row_newbcast:" I " row_mask:0xf bank_mask:0xf"
// two output degrees of a translation: re0 += t0 x, im0 += t0 y, re1 += t1 x, im1 += t1 y
template <int I>
__device__ __forceinline__ void tr4_bc(double& re0, double& im0, double& re1, double& im1, double c, double x, double y)
{
    asm("v_fmac_f64_dpp %0, %4, %5" LFMM_BC("%7") "\n\tv_fmac_f64_dpp %1, %4, %6" LFMM_BC("%7")
        "\n\tv_fmac_f64_dpp %2, %4, %5" LFMM_BC("%8") "\n\tv_fmac_f64_dpp %3, %4, %6" LFMM_BC("%8")
        : "+&v"(re0), "+&v"(im0), "+&v"(re1), "+&v"(im1)
        : "v"(c), "v"(x), "v"(y), "n"(I), "n"(I + 1));
}
#undef LFMM_BC

}  // namespace lfmm
