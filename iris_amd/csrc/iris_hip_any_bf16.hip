// The any-shape kernel for bf16 inputs (see any_kernel.h).
#include "any_kernel.h"

template int dispatch_any<IN_BF16, ElemBF16>(const FusedParams&, int, int, hipStream_t, const char*, int);
template int dispatch_any<IN_BF16, ElemF32>(const FusedParams&, int, int, hipStream_t, const char*, int);
