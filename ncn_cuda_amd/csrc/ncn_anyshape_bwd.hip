// The reversible backward of ncn_anyshape.hip.
#define NCN_ANYSHAPE_BACKWARD 1
#include "ncn_anyshape.hip"
