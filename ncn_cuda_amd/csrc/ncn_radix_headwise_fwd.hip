// Radix kernels of one kind; see ncn_radix_build.hip.
#define NCN_RADIX_HEADWISE true
#include "ncn_radix_build.hip"
