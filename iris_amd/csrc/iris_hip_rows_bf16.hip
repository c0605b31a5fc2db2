// libiris_hip: the MFMA kernel builds for bf16 inputs and outputs whose rows start and end anywhere.
#include "fused_kernel.h"

template int dispatch_mfma_rows<IN_BF16>(const FusedParams&, int, bool, int, hipStream_t);
