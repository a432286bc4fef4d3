// The backward stage kernels for bfloat16 launches with a wave for every tile (see ncn_bwd.hip).
#define NCN_TYPES_BUILD kBf16Types
#include "ncn_bwd.hip"
