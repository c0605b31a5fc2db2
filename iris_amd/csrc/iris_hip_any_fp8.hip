// The any-shape kernel for e4m3 inputs (see any_kernel.h).
#include "any_kernel.h"

template int dispatch_any<IN_FP8, ElemBF16>(const FusedParams&, int, int, hipStream_t, const char*, int);
template int dispatch_any<IN_FP8, ElemF16>(const FusedParams&, int, int, hipStream_t, const char*, int);
