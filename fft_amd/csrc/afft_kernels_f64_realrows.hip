// FP64 row passes with a real pass.
#define AFGPU_PART 3
#include "afft_kernels_f64.hip"
