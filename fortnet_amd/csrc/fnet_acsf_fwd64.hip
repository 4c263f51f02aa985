// The FP64 forward instances of the ACSF kernels (fnet_acsf.hip).
#define FNET_ACSF_PART 2
#include "fnet_acsf.hip"
