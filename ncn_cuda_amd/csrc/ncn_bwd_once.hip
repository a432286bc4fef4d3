// The backward stage kernels of every element type and activation for launches with a wave for every tile (see ncn_bwd.hip).
#define NCN_TYPES_BUILD kAnyTypesOnce
#include "ncn_bwd.hip"
