// The backward stage kernels for bfloat16 launches that carry a grouping table or context lengths, with a wave for every
// tile (see ncn_bwd.hip).
#define NCN_INDEXED_BUILD 1
#define NCN_TYPES_BUILD kBf16Types
#include "ncn_bwd.hip"
