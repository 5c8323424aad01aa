// smx_split_ops.h -- host launchers of the two-launch step (smx_split.h).  The definitions are in
// smx_split_launch.h, instantiated per precision in smx_split_z_*.hip and smx_split_x_*.hip.
#pragma once
#include "smx_split_adv.h"
#include "smx_split_neu.h"
#include "smx_split_surf.h"

namespace smx {

// Whether the two kernels exist for this grid: ny has a split and both tiles fit a workgroup.
template <typename T> bool split_z_fits(int ny, int nz);
template <typename T> bool split_x_fits(int nx, int ny);
template <typename T> int split_x_blocks(int nx, int ny, int nz);  // of one step (0: none)

// Blocks of the z kernel that take a tile each (one FP64 partial per block).
template <typename T> int split_z_blocks(const PParams<T>& p);
template <typename T> hipError_t split_z(const SplitArgs<T>& s, int op, hipStream_t st);
template <typename T> hipError_t split_x(const SplitArgs<T>& s, hipStream_t st);
// One launch for nbox boxes of one grid (arguments in device memory).
template <typename T>
hipError_t split_z_grp(const SplitArgs<T>* g, int nbox, const PParams<T>& p, int op, hipStream_t st);
template <typename T> hipError_t split_x_grp(const SplitArgs<T>* g, int nbox, const PParams<T>& p, hipStream_t st);
// FP64 real field of a split-form stage array of type TI.
template <typename TI>
hipError_t split_real(const cplx<TI>* a, double* out, const PParams<double>& p, hipStream_t st);
// The advected step's four launches (smx_split_adv.h).
template <typename T> bool split_adv_fits_z(int ny, int nz);
template <typename T> bool split_adv_fits_x(int nx, int ny);
template <typename T> hipError_t split_adv_force(const SplitAdvArgs<T>& s, hipStream_t st);
template <typename T> hipError_t split_adv_stokes(const SplitAdvArgs<T>& s, hipStream_t st);
template <typename T> hipError_t split_adv_advnl(const SplitAdvArgs<T>& s, hipStream_t st);
template <typename T> hipError_t split_adv_update(const SplitAdvArgs<T>& s, hipStream_t st);
bool split_real_fits(int ny, int nz);
// surfTrack's psi, scan and z derivative from a split-form stage array (smx_split_surf.h); hipErrorNotSupported
// for a grid whose tile does not take it.
template <typename TI>
hipError_t split_scan_surf(const cplx<TI>* a, const PParams<double>& p, const SplitScan& s, hipStream_t st);
template <typename TI>
hipError_t nsplit_scan_surf(const cplx<TI>* a, const PParams<double>& p, const cplx<double>* qtz, const SplitScan& s,
                            hipStream_t st);
// The Neumann step's two launches, its real field and its change of form (smx_split_neu.h).
template <typename T> bool nsplit_z_fits(int nx, int ny, int nz);
template <typename T> bool nsplit_x_fits(int nx, int ny);
template <typename T> int nsplit_z_per_cu(int nx, int ny, int nz);  // blocks whose tiles fit a CU (0: none)
template <typename T> int nsplit_x_per_cu(int nx, int ny);
template <typename T> int nsplit_z_blocks(const PParams<T>& p);
template <typename T> hipError_t nsplit_z(const SplitNeuArgs<T>& s, hipStream_t st);
template <typename T> hipError_t nsplit_x(const SplitNeuArgs<T>& s, hipStream_t st);
bool nsplit_real_fits(int nx, int ny, int nz);
template <typename TI>
hipError_t nsplit_real(const cplx<TI>* a, double* out, const PParams<double>& p, const cplx<double>* qtz, hipStream_t st);
template <typename TI, typename TO>
hipError_t nsplit_form(const TI* in, TO* out, int nx, int ny, int nz, const cplx<double>* twy, const cplx<double>* qty,
                       int dir, hipStream_t st);
// Rows of a stage array (or, with the perm directions, of the carry) between the two forms, in place
// allowed.  kmul: k_y table of the d/dy of a standard-form input, or nullptr.
template <typename T>
hipError_t split_form(const cplx<T>* in, cplx<T>* out, int64_t nrows, int ny, const cplx<T>* twy, int dir,
                      const T* kmul, hipStream_t st);
// To the standard form from rows of type TI (in place allowed for TI = T).
template <typename T, typename TI>
hipError_t split_form_std(const cplx<TI>* in, cplx<T>* out, int64_t nrows, int ny, const cplx<T>* twy,
                          hipStream_t st);

}  // namespace smx
