// The FP32-only form of the split-FP32 doubles kernels (no corrections).
#define ATRIP_SPLIT_CORR false
#define ATRIP_SPLIT_LAUNCH launch_doubles_fp32
#include "doubles_split.hip"
