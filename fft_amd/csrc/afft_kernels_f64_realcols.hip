// FP64 column passes with a real pass.
#define AFGPU_PART 2
#include "afft_kernels_f64.hip"
