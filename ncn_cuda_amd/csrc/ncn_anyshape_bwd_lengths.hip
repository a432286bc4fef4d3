// The reversible backward of ncn_anyshape.hip for launches with context lengths.
#define NCN_ANYSHAPE_BACKWARD 1
#define NCN_ANYSHAPE_LENGTHS 1
#include "ncn_anyshape.hip"
