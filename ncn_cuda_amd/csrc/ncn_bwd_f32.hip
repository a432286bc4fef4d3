// The backward stage kernels for float32 launches with a wave for every tile (see ncn_bwd.hip).
#define NCN_TYPES_BUILD kF32Types
#include "ncn_bwd.hip"
