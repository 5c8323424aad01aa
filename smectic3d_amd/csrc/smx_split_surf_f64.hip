// Instantiates surfTrack's scans of split-form arrays of type double.
#define SMX_SPLIT_SURF
#include "smx_split_launch.h"
template hipError_t smx::split_scan_surf<double>(const smx::cplx<double>*, const smx::PParams<double>&, const smx::SplitScan&,
                                             hipStream_t);
template hipError_t smx::nsplit_scan_surf<double>(const smx::cplx<double>*, const smx::PParams<double>&,
                                              const smx::cplx<double>*, const smx::SplitScan&, hipStream_t);
