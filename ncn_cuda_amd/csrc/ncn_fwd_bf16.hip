// The forward and inverse stage kernels for bfloat16 launches (see ncn_fwd.hip).
#define NCN_TYPES_BUILD kBf16Types
#include "ncn_fwd.hip"
