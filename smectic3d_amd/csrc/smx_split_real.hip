// Instantiates the real-field inverse of split-form stage arrays.
#define SMX_SPLIT_REAL
#include "smx_split_launch.h"
template hipError_t smx::split_real<float>(const smx::cplx<float>*, double*, const smx::PParams<double>&, hipStream_t);
template hipError_t smx::split_real<double>(const smx::cplx<double>*, double*, const smx::PParams<double>&, hipStream_t);
