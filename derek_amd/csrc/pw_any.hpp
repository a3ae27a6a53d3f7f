// Pruned-FFT passes for every length n = r1 * r2 with radices up to 16 (see
// pw_any.hip): the forms of pw_fft.hpp's passes for the lengths without
// kernels of their own.  Each launcher returns false where the length has no
// such split or the tile does not fit the LDS; the caller then takes the
// Stockham kernels.
#pragma once
#include "pw_fft.hpp"

namespace derek {

template <typename R>
bool any_z_inv(const PwBatch& B, PwBlock<R> psi, const Axis<R>& az, cx_t<R>* S, bool zmajor, hipStream_t s);
template <typename R>
bool any_z_fwd(const PwBatch& B, const cx_t<R>* S, const Axis<R>& az, PwBlock<R> psi, PwBlock<R> hpsi, bool zmajor,
               hipStream_t s);
template <typename R>
bool any_y(const PwBatch& B, cx_t<R>* S, cx_t<R>* P, const Axis<R>& ay, int nz, int sign, int bands_per_wg,
           hipStream_t s);
template <typename R>
bool any_x_vmul(const PwBatch& B, cx_t<R>* P, const Axis<R>& ax, int64_t nyz, const R* vloc, R vscale,
                int bands_per_wg, hipStream_t s);
template <typename R>
bool any_x_density(const PwBatch& B, const cx_t<R>* P, const Axis<R>& ax, int64_t nyz, const double* occ, int occ_ks,
                   double* rho, int keep, hipStream_t s);

}  // namespace derek
