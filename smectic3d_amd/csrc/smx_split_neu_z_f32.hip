// Instantiates the z kernels of the two-launch Neumann step for float.
#define SMX_SPLIT_NEU_Z
#include "smx_split_launch.h"
template bool smx::nsplit_z_fits<float>(int, int, int);
template int smx::nsplit_z_blocks<float>(const smx::PParams<float>&);
template hipError_t smx::nsplit_z<float>(const smx::SplitNeuArgs<float>&, hipStream_t);
