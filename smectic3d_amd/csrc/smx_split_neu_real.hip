// Instantiates the real field and the change of form of Neumann split-form arrays.
#define SMX_SPLIT_NEU_REAL
#include "smx_split_launch.h"
using smx::cplx;
template hipError_t smx::nsplit_real<float>(const cplx<float>*, double*, const smx::PParams<double>&,
                                            const cplx<double>*, hipStream_t);
template hipError_t smx::nsplit_real<double>(const cplx<double>*, double*, const smx::PParams<double>&,
                                             const cplx<double>*, hipStream_t);
#define SMX_NFORM(TI, TO)                                                                                   \
  template hipError_t smx::nsplit_form<TI, TO>(const TI*, TO*, int, int, int, const cplx<double>*,         \
                                               const cplx<double>*, int, hipStream_t);
SMX_NFORM(float, float)
SMX_NFORM(float, double)
SMX_NFORM(double, double)
