// Instantiates the x kernels of the two-launch step and the change of form for double.
#define SMX_SPLIT_X
#include "smx_split_launch.h"
template bool smx::split_x_fits<double>(int, int);
template int smx::split_x_blocks<double>(int, int, int);
template hipError_t smx::split_x<double>(const smx::SplitArgs<double>&, hipStream_t);
template hipError_t smx::split_x_grp<double>(const smx::SplitArgs<double>*, int, const smx::PParams<double>&, hipStream_t);
template hipError_t smx::split_form<double>(const smx::cplx<double>*, smx::cplx<double>*, int64_t, int, const smx::cplx<double>*,
                                           int, const double*, hipStream_t);
template hipError_t smx::split_form_std<double, float>(const smx::cplx<float>*, smx::cplx<double>*, int64_t, int,
                                                       const smx::cplx<double>*, hipStream_t);
