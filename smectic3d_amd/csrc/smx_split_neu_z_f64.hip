// Instantiates the z kernels of the two-launch Neumann step for double.
#define SMX_SPLIT_NEU_Z
#include "smx_split_launch.h"
template bool smx::nsplit_z_fits<double>(int, int, int);
template int smx::nsplit_z_blocks<double>(const smx::PParams<double>&);
template hipError_t smx::nsplit_z<double>(const smx::SplitNeuArgs<double>&, hipStream_t);
template int smx::nsplit_z_per_cu<double>(int, int, int);
