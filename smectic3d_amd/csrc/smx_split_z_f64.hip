// Instantiates the z kernels of the two-launch step for double.
#define SMX_SPLIT_Z
#include "smx_split_launch.h"
template bool smx::split_z_fits<double>(int, int);
template int smx::split_z_blocks<double>(const smx::PParams<double>&);
template hipError_t smx::split_z<double>(const smx::SplitArgs<double>&, int, hipStream_t);
template hipError_t smx::split_z_grp<double>(const smx::SplitArgs<double>*, int, const smx::PParams<double>&, int, hipStream_t);
