// Radix kernels of one kind; see ncn_radix_build.hip.
#define NCN_RADIX_HEADWISE true
#define NCN_RADIX_TANH false
#include "ncn_radix_build.hip"
