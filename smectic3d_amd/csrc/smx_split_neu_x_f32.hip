// Instantiates the x kernels of the two-launch Neumann step for float.
#define SMX_SPLIT_NEU_X
#include "smx_split_launch.h"
template bool smx::nsplit_x_fits<float>(int, int);
template hipError_t smx::nsplit_x<float>(const smx::SplitNeuArgs<float>&, hipStream_t);
