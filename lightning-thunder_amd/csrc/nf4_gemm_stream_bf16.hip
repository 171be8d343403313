#define STREAM_F16 false
#define STREAM_NESTED false
#define STREAM_LAUNCH launch_bf16
#include "nf4_gemm_stream_kernels.h"
