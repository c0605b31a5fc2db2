// libiris_hip: the kernel for small outputs, builds for bf16 inputs (see decode_kernel.h).
#include "decode_kernel.h"

template int dispatch_decode<IN_BF16>(FusedParams&, bool, int, int, hipStream_t);
