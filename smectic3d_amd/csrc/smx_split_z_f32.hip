// Instantiates the z kernels of the two-launch step for float.
#define SMX_SPLIT_Z
#include "smx_split_launch.h"
template bool smx::split_z_fits<float>(int, int);
template int smx::split_z_blocks<float>(const smx::PParams<float>&);
template hipError_t smx::split_z<float>(const smx::SplitArgs<float>&, int, hipStream_t);
template hipError_t smx::split_z_grp<float>(const smx::SplitArgs<float>*, int, const smx::PParams<float>&, int, hipStream_t);
