// Instantiates the x kernels of the advected step in four launches for float.
#define SMX_SPLIT_ADV_X
#include "smx_split_launch.h"
template bool smx::split_adv_fits_x<float>(int, int);
template hipError_t smx::split_adv_stokes<float>(const smx::SplitAdvArgs<float>&, hipStream_t);
template hipError_t smx::split_adv_update<float>(const smx::SplitAdvArgs<float>&, hipStream_t);
