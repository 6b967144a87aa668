// instances.hip -- the transform kernels of the compiled length RPCF_LENGTH (instances.hpp).
#include "instances.hpp"

RPCF_INSTANCES(, RPCF_LENGTH)
