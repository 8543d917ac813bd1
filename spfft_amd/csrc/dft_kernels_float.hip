// FP32 transforms of the matrix kernels (see dft_kernels.hip).
#define SPFFT_DFT_FLOAT 1
#include "dft_kernels.hip"
