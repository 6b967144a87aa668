// instances.hip -- the transform kernels of the compiled length RPCF_LENGTH (instances.hpp); with
// RPCF_XY_ONLY its FP64 x and span transforms alone, with RPCF_SPAN_ONLY its span transforms.
#include "instances.hpp"

#if defined(RPCF_XY_ONLY)
RPCF_INSTANCES_XY(, RPCF_LENGTH, double)
#elif defined(RPCF_SPAN_ONLY)
RPCF_INSTANCES_SPAN(, RPCF_LENGTH, double)
RPCF_INSTANCES_SPAN(, RPCF_LENGTH, float)
#else
RPCF_INSTANCES(, RPCF_LENGTH)
#endif
