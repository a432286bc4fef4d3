// The forward and inverse of ncn_anyshape.hip for launches with context lengths.
#define NCN_ANYSHAPE_LENGTHS 1
#include "ncn_anyshape.hip"
