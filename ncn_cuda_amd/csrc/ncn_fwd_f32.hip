// The forward and inverse stage kernels for float32 launches (see ncn_fwd.hip).
#define NCN_TYPES_BUILD kF32Types
#include "ncn_fwd.hip"
