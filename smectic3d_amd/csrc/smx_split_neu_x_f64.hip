// Instantiates the x kernels of the two-launch Neumann step for double.
#define SMX_SPLIT_NEU_X
#include "smx_split_launch.h"
template bool smx::nsplit_x_fits<double>(int, int);
template hipError_t smx::nsplit_x<double>(const smx::SplitNeuArgs<double>&, hipStream_t);
template int smx::nsplit_x_per_cu<double>(int, int);
