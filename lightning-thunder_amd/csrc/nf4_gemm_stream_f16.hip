#define STREAM_F16 true
#define STREAM_NESTED false
#define STREAM_LAUNCH launch_f16
#include "nf4_gemm_stream_kernels.h"
