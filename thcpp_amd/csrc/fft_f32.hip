// FP32 transforms of fft.hip, in a unit of their own: the kernels of the two
// precisions take over a minute each to compile and compile side by side.
#define THC_FFT_F32
#include "fft.hip"
