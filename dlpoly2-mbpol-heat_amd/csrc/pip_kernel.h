// pip_kernel.h -- the MB-pol polynomials (2-body poly_2b_v6x, 31 variables, 1153 basis polynomials,
// poly-2b-v6x.h; 3-body poly_3b_v2x, 36 variables, 1163 basis polynomials, poly-3b-v2x.h:10-17) as
// sliced straight-line code generated by gen_pip.py, one kernel for both.
//
// One wavefront evaluates one slice of a polynomial for 64 clusters.  Each lane keeps its variables
// and partial gradients in VGPRs (164 VGPRs in FP64, no scratch); coefficients arrive through scalar
// loads.  The blocks of a slice are consecutive, so that a CU's wavefronts run the same code (a slice
// is some 50 KB of instructions), and the trimers' come first, being the longer; the dimers'
// fill in beside them instead of taking a launch of their own (9 waters: 40 + 16 us -> 40).
#pragma once
#include "mbgpu_internal.h"
#include "gen/pip2b_gen.inc"
#include "gen/pip3b_gen.inc"

template <typename T>
__global__ __launch_bounds__(64) void k_pip(const int* __restrict__ counts, const T* __restrict__ xv2,
                                            T* __restrict__ part2, int cap2, const T* __restrict__ cs2,
                                            const T* __restrict__ xv3, T* __restrict__ part3, int cap3,
                                            const T* __restrict__ cs3)
{
    // clusters below the count (device memory) of a buffer laid out with stride cap
    const int nb2 = (cap2 + 63) / 64, nb3 = (cap3 + 63) / 64;
    int b = blockIdx.x;
    if (b < nb3 * PIP3B_NSLICES) {
        const int c = (b % nb3) * 64 + threadIdx.x;
        if (c < min(counts[1], cap3)) pip3b_slice<T>(b / nb3, xv3, part3, c, cap3, cs3);
    } else {
        b -= nb3 * PIP3B_NSLICES;
        const int c = (b % nb2) * 64 + threadIdx.x;
        if (c < min(counts[0], cap2)) pip2b_slice<T>(b / nb2, xv2, part2, c, cap2, cs2);
    }
}

template <typename T>
void launch_pip(const int* counts, const T* xv2, T* part2, int cap2, const T* cs2, const T* xv3, T* part3, int cap3,
                const T* cs3, hipStream_t s)
{
    const int nb = (cap3 + 63) / 64 * PIP3B_NSLICES + (cap2 + 63) / 64 * PIP2B_NSLICES;
    if (nb > 0)
        hipLaunchKernelGGL(k_pip<T>, dim3(nb), dim3(64), 0, s, counts, xv2, part2, cap2, cs2, xv3, part3, cap3, cs3);
}
