// FP32 plain and twiddled column passes.
#define AFGPU_PART 1
#include "afft_kernels_f32.hip"
