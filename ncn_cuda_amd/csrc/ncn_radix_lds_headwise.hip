// ncn_radix_lds.hip for heads of one feature.
#define NCN_RADIX_HEADWISE true
#include "ncn_radix_lds.hip"
