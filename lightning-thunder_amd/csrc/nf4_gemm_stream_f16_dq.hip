#define STREAM_F16 true
#define STREAM_NESTED true
#define STREAM_LAUNCH launch_f16_dq
#include "nf4_gemm_stream_kernels.h"
