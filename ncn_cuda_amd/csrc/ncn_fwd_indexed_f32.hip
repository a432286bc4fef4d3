// The forward and inverse stage kernels for float32 launches that carry a grouping table or context lengths (see
// ncn_fwd.hip).
#define NCN_INDEXED_BUILD 1
#define NCN_TYPES_BUILD kF32Types
#include "ncn_fwd.hip"
