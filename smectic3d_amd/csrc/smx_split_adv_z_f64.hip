// Instantiates the z kernels of the advected step in four launches for double.
#define SMX_SPLIT_ADV_Z
#include "smx_split_launch.h"
template bool smx::split_adv_fits_z<double>(int, int);
template hipError_t smx::split_adv_force<double>(const smx::SplitAdvArgs<double>&, hipStream_t);
template hipError_t smx::split_adv_advnl<double>(const smx::SplitAdvArgs<double>&, hipStream_t);
