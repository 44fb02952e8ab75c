// pip_f64.hip -- the MB-pol polynomials in FP64 and the tables of their generated code.
#include "pip_kernel.h"

void launch_pip_f64(const int* counts, const double* xv2, double* part2, int cap2, const double* cs2, const double* xv3,
                    double* part3, int cap3, const double* cs3, hipStream_t s)
{
    launch_pip(counts, xv2, part2, cap2, cs2, xv3, part3, cap3, cs3, s);
}

int pip2b_nslices() { return PIP2B_NSLICES; }
int pip2b_stream_len() { return PIP2B_STREAM_LEN; }
const short* pip2b_stream_table() { return pip2b_stream_basis; }
const double* pip2b_stream_values() { return pip2b_stream_coef; }
int pip3b_nslices() { return PIP3B_NSLICES; }
int pip3b_stream_len() { return PIP3B_STREAM_LEN; }
const short* pip3b_stream_table() { return pip3b_stream_basis; }
const double* pip3b_stream_values() { return pip3b_stream_coef; }
