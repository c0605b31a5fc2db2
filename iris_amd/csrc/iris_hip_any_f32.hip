// The any-shape kernel for float32 inputs (see any_kernel.h).
#include "any_kernel.h"

template int dispatch_any<IN_F32, ElemF32>(const FusedParams&, int, int, hipStream_t, const char*, int);
