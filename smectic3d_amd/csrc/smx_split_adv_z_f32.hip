// Instantiates the z kernels of the advected step in four launches for float.
#define SMX_SPLIT_ADV_Z
#include "smx_split_launch.h"
template bool smx::split_adv_fits_z<float>(int, int);
template hipError_t smx::split_adv_force<float>(const smx::SplitAdvArgs<float>&, hipStream_t);
template hipError_t smx::split_adv_advnl<float>(const smx::SplitAdvArgs<float>&, hipStream_t);
