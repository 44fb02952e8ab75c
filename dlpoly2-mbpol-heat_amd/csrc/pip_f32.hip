// pip_f32.hip -- the MB-pol polynomials in FP32 (mixed-precision mode).
#include "pip_kernel.h"

void launch_pip_f32(const int* counts, const float* xv2, float* part2, int cap2, const float* cs2, const float* xv3,
                    float* part3, int cap3, const float* cs3, hipStream_t s)
{
    launch_pip(counts, xv2, part2, cap2, cs2, xv3, part3, cap3, cs3, s);
}
