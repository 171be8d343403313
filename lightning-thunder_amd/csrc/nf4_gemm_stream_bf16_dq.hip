#define STREAM_F16 false
#define STREAM_NESTED true
#define STREAM_LAUNCH launch_bf16_dq
#include "nf4_gemm_stream_kernels.h"
