// instances.hip -- the transform kernels of the compiled length RPCF_LENGTH (instances.hpp); with
// RPCF_XY_ONLY its FP64 x and span transforms alone.
#include "instances.hpp"

#ifdef RPCF_XY_ONLY
RPCF_INSTANCES_XY(, RPCF_LENGTH, double)
#else
RPCF_INSTANCES(, RPCF_LENGTH)
#endif
