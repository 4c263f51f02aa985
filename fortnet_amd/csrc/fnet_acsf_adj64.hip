// The FP64 adjoint instances of the ACSF kernels (fnet_acsf.hip).
#define FNET_ACSF_PART 3
#include "fnet_acsf.hip"
