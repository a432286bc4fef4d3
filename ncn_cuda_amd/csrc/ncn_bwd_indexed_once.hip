// The same for launches that carry a grouping table or context lengths (see ncn_bwd.hip).
#define NCN_INDEXED_BUILD 1
#define NCN_TYPES_BUILD kAnyTypesOnce
#include "ncn_bwd.hip"
