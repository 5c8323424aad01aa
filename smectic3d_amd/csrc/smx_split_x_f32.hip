// Instantiates the x kernels of the two-launch step and the change of form for float.
#define SMX_SPLIT_X
#include "smx_split_launch.h"
template bool smx::split_x_fits<float>(int, int);
template hipError_t smx::split_x<float>(const smx::SplitArgs<float>&, hipStream_t);
template hipError_t smx::split_x_grp<float>(const smx::SplitArgs<float>*, int, const smx::PParams<float>&, hipStream_t);
template hipError_t smx::split_form<float>(const smx::cplx<float>*, smx::cplx<float>*, int64_t, int, const smx::cplx<float>*,
                                           int, const float*, hipStream_t);
