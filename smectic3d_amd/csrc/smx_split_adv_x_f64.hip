// Instantiates the x kernels of the advected step in four launches for double.
#define SMX_SPLIT_ADV_X
#include "smx_split_launch.h"
template bool smx::split_adv_fits_x<double>(int, int);
template hipError_t smx::split_adv_stokes<double>(const smx::SplitAdvArgs<double>&, hipStream_t);
template hipError_t smx::split_adv_update<double>(const smx::SplitAdvArgs<double>&, hipStream_t);
