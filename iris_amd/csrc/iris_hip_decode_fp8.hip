// libiris_hip: the kernel for small outputs, builds for fp8 inputs (see decode_kernel.h).
#include "decode_kernel.h"

template int dispatch_decode<IN_FP8>(FusedParams&, bool, int, int, hipStream_t);
