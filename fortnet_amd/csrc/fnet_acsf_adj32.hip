// The FP32 adjoint instances of the ACSF kernels (fnet_acsf.hip).
#define FNET_ACSF_PART 1
#include "fnet_acsf.hip"
