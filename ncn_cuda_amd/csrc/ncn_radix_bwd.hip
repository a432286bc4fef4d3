// Radix kernels of one kind; see ncn_radix_build.hip.
#define NCN_RADIX_BACKWARD true
#include "ncn_radix_build.hip"
