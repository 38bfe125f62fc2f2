// FP64 plain and twiddled column passes.
#define AFGPU_PART 1
#include "afft_kernels_f64.hip"
