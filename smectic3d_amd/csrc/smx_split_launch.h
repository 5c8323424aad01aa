// smx_split_launch.h -- runtime-length dispatch of the two-launch step's kernels.
#pragma once
#include "smx_launch.h"
#include "smx_split_ops.h"

namespace smx {

// f(IC<L>, IC<RA>) for a z length and a y split, f(IC<L>, IC<RB>) for an x length and a y split.
template <typename F>
hipError_t split_z_dispatch(int nz, int ra, F&& f) {
#define SMX_CASE(L)                          \
  if (nz == L) {                             \
    switch (ra) {                            \
      case 4: return f(IC<L>{}, IC<4>{});    \
      case 8: return f(IC<L>{}, IC<8>{});    \
      case 12: return f(IC<L>{}, IC<12>{});  \
      case 16: return f(IC<L>{}, IC<16>{});  \
      case 24: return f(IC<L>{}, IC<24>{});  \
      default: return hipErrorInvalidValue;  \
    }                                        \
  }
  SMX_FOR_EACH_LENGTH(SMX_CASE)
#undef SMX_CASE
  return hipErrorInvalidValue;
}
template <typename F>
hipError_t split_x_dispatch(int nx, int rb, F&& f) {
#define SMX_CASE(L)                          \
  if (nx == L) {                             \
    switch (rb) {                            \
      case 4: return f(IC<L>{}, IC<4>{});    \
      case 8: return f(IC<L>{}, IC<8>{});    \
      case 12: return f(IC<L>{}, IC<12>{});  \
      case 16: return f(IC<L>{}, IC<16>{});  \
      default: return hipErrorInvalidValue;  \
    }                                        \
  }
  SMX_FOR_EACH_LENGTH(SMX_CASE)
#undef SMX_CASE
  return hipErrorInvalidValue;
}

// The y lengths with a division (split_ra, nsplit_ra).
#define SMX_FOR_EACH_SPLIT(X) X(16) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384)

// f(ZS of the grid): the tile with whole pieces where split_whole asks for it and there are blocks enough.  One
// choice for a box, alone or in a group, so that its partial sums are counted alike.
template <typename T, int L, int RA, typename F>
hipError_t split_z_tile(int nx, int ny, F&& f) {
  if constexpr (split_whole<T>(L, RA)) {
    using Z = ZS<T, L, RA, kSplitYC>;
    static_assert(Z::fits, "both tiles fit");
    if (nx * (ny / RA / kSplitYC) >= kSplitWholeBlocks) return f(Z{});
  }
  return f(ZS<T, L, RA>{});
}

// Blocks that project the carry: 8 pairs' entries per thread.
template <typename Z, typename T>
static int split_nproj(const PParams<T>& p) {
  return (int)((2 * p.nxy + 8 * Z::NT - 1) / (8 * Z::NT));
}

#ifdef SMX_SPLIT_Z
template <typename T>
bool split_z_fits(int ny, int nz) {
  const int ra = split_ra(ny);
  return ra != 0 && split_z_dispatch(nz, ra, [&](auto l, auto r) -> hipError_t {
           using Z = ZS<T, decltype(l)::value, decltype(r)::value>;
           return Z::fits && (ny / ra) % Z::NY2 == 0 ? hipSuccess : hipErrorInvalidValue;
         }) == hipSuccess;
}
template <typename T>
int split_z_blocks(const PParams<T>& p) {
  int n = 0;
  const int ra = split_ra(p.ny);
  (void)split_z_dispatch(p.nz, ra, [&](auto l, auto r) -> hipError_t {
    return split_z_tile<T, decltype(l)::value, decltype(r)::value>(p.nx, p.ny, [&](auto z) -> hipError_t {
      n = p.nx * (p.ny / ra / decltype(z)::NY2);
      return hipSuccess;
    });
  });
  return n;
}
template <typename T>
hipError_t split_z(const SplitArgs<T>& s, int op, hipStream_t st) {
  return split_z_dispatch(s.p.nz, split_ra(s.p.ny), [&](auto l, auto r) -> hipError_t {
    return split_z_tile<T, decltype(l)::value, decltype(r)::value>(s.p.nx, s.p.ny, [&](auto z) -> hipError_t {
      using Z = decltype(z);
      if constexpr (!Z::fits) {
        return hipErrorInvalidValue;
      } else {
        const int np = split_nproj<Z>(s.p);
        SMX_LAUNCH((k_zsplit<Z>), dim3((unsigned)(np + split_z_blocks(s.p))), dim3(Z::NT), 0, st, s, op, np);
        return hipGetLastError();
      }
    });
  });
}
template <typename T>
hipError_t split_z_grp(const SplitArgs<T>* g, int nbox, const PParams<T>& p, int op, hipStream_t st) {
  if (nbox < 1 || nbox > 65535) return hipErrorInvalidValue;
  return split_z_dispatch(p.nz, split_ra(p.ny), [&](auto l, auto r) -> hipError_t {
    return split_z_tile<T, decltype(l)::value, decltype(r)::value>(p.nx, p.ny, [&](auto z) -> hipError_t {
      using Z = decltype(z);
      if constexpr (!Z::fits) {
        return hipErrorInvalidValue;
      } else {
        const int np = split_nproj<Z>(p);
        SMX_LAUNCH((k_zsplit_grp<Z>), dim3((unsigned)(np + split_z_blocks(p)), (unsigned)nbox), dim3(Z::NT), 0, st,
                   g, op, np);
        return hipGetLastError();
      }
    });
  });
}
#endif

#ifdef SMX_SPLIT_ADV_Z
template <typename T>
bool split_adv_fits_z(int ny, int nz) {
  const int ra = split_ra(ny);
  return ra != 0 && split_z_dispatch(nz, ra, [&](auto l, auto r) -> hipError_t {
           using Z = ZS<T, decltype(l)::value, decltype(r)::value>;
           return zsa_fits<Z>() && (ny / ra) % Z::NY2 == 0 ? hipSuccess : hipErrorInvalidValue;
         }) == hipSuccess;
}
template <typename T>
hipError_t split_adv_force(const SplitAdvArgs<T>& s, hipStream_t st) {
  const PParams<T>& p = s.ap.p;
  return split_z_dispatch(p.nz, split_ra(p.ny), [&](auto l, auto r) -> hipError_t {
    return split_z_tile<T, decltype(l)::value, decltype(r)::value>(p.nx, p.ny, [&](auto z) -> hipError_t {
      using Z = decltype(z);
      if constexpr (!zsa_fits<Z>()) {
        return hipErrorInvalidValue;
      } else {
        const int np = split_nproj<Z>(p), nb = p.nx * (p.ny / Z::RA / Z::NY2);
        SMX_LAUNCH((k_zsplit_force<Z>), dim3((unsigned)(np + nb)), dim3(Z::NT), 0, st, s, np);
        return hipGetLastError();
      }
    });
  });
}
template <typename T>
hipError_t split_adv_advnl(const SplitAdvArgs<T>& s, hipStream_t st) {
  const PParams<T>& p = s.ap.p;
  return split_z_dispatch(p.nz, split_ra(p.ny), [&](auto l, auto r) -> hipError_t {
    return split_z_tile<T, decltype(l)::value, decltype(r)::value>(p.nx, p.ny, [&](auto z) -> hipError_t {
      using Z = decltype(z);
      if constexpr (!zsa_fits<Z>()) {
        return hipErrorInvalidValue;
      } else {
        SMX_LAUNCH((k_zsplit_advnl<Z>), dim3((unsigned)(p.nx * (p.ny / Z::RA / Z::NY2))), dim3(Z::NT), 0, st, s);
        return hipGetLastError();
      }
    });
  });
}
#endif

#ifdef SMX_SPLIT_ADV_X
template <typename T>
bool split_adv_fits_x(int nx, int ny) {
  const int ra = split_ra(ny);
  return ra != 0 && split_x_dispatch(nx, ny / ra, [&](auto l, auto r) -> hipError_t {
           using X = XS<T, decltype(l)::value, decltype(r)::value>;
           return xsa_fits<X>() && ny % X::NC == 0 ? hipSuccess : hipErrorInvalidValue;
         }) == hipSuccess;
}
template <typename T>
hipError_t split_adv_stokes(const SplitAdvArgs<T>& s, hipStream_t st) {
  const PParams<T>& p = s.ap.p;
  return split_x_dispatch(p.nx, p.ny / split_ra(p.ny), [&](auto l, auto r) -> hipError_t {
    using X = XS<T, decltype(l)::value, decltype(r)::value>;
    if constexpr (!xsa_fits<X>()) {
      return hipErrorInvalidValue;
    } else {
      SMX_LAUNCH((k_xsplit_stokes<X>), dim3((unsigned)(p.ny / X::NC * p.nzh)), dim3(X::NT), 0, st, s);
      return hipGetLastError();
    }
  });
}
template <typename T>
hipError_t split_adv_update(const SplitAdvArgs<T>& s, hipStream_t st) {
  const PParams<T>& p = s.ap.p;
  return split_x_dispatch(p.nx, p.ny / split_ra(p.ny), [&](auto l, auto r) -> hipError_t {
    using X = XS<T, decltype(l)::value, decltype(r)::value>;
    if constexpr (!xsa_fits<X>()) {
      return hipErrorInvalidValue;
    } else {
      const unsigned nb = (unsigned)(p.ny / X::NC * p.nzh);
      if constexpr (sizeof(T) == 4 && X::L >= 384) {
        if (nb > 256) {
          SMX_LAUNCH((k_xsplit_adv<X, true>), dim3(nb), dim3(X::NT), 0, st, s);
          return hipGetLastError();
        }
      }
      SMX_LAUNCH((k_xsplit_adv<X, false>), dim3(nb), dim3(X::NT), 0, st, s);
      return hipGetLastError();
    }
  });
}
#endif

#ifdef SMX_SPLIT_REAL
bool split_real_fits(int ny, int nz) {
  const int ra = split_ra(ny);
  return ra != 0 && split_z_dispatch(nz, ra, [&](auto l, auto r) -> hipError_t {
           using Z = ZS<double, decltype(l)::value, decltype(r)::value>;
           return Z::fits && (size_t)(Z::SLDS + Z::L) * sizeof(cplx<double>) <= 160 * 1024 && (ny / ra) % Z::NY2 == 0
                      ? hipSuccess
                      : hipErrorInvalidValue;
         }) == hipSuccess;
}
template <typename TI>
hipError_t split_real(const cplx<TI>* a, double* out, const PParams<double>& p, hipStream_t st) {
  return split_z_dispatch(p.nz, split_ra(p.ny), [&](auto l, auto r) -> hipError_t {
    constexpr int L = decltype(l)::value, RA = decltype(r)::value;
    using Z = ZS<double, L, RA>;
    if constexpr (!Z::fits) {
      return hipErrorInvalidValue;
    } else {
      SMX_LAUNCH((k_zsplit_real<Z, TI>), dim3((unsigned)(p.nx * (p.ny / RA / Z::NY2))), dim3(Z::NT), 0, st, a, out,
                 p);
      return hipGetLastError();
    }
  });
}
#endif

#ifdef SMX_SPLIT_X
template <typename T>
bool split_x_fits(int nx, int ny) {
  const int ra = split_ra(ny);
  return ra != 0 && split_x_dispatch(nx, ny / ra, [&](auto l, auto r) -> hipError_t {
           using X = XS<T, decltype(l)::value, decltype(r)::value>;
           return X::fits && ny % X::NC == 0 ? hipSuccess : hipErrorInvalidValue;
         }) == hipSuccess;
}
template <typename T>
int split_x_blocks(int nx, int ny, int nz) {
  const int ra = split_ra(ny);
  int n = 0;
  if (ra != 0)
    (void)split_x_dispatch(nx, ny / ra, [&](auto l, auto r) -> hipError_t {
      n = ny / XS<T, decltype(l)::value, decltype(r)::value>::NC * (nz / 2 + 1);
      return hipSuccess;
    });
  return n;
}
template <typename T>
hipError_t split_x(const SplitArgs<T>& s, hipStream_t st) {
  return split_x_dispatch(s.p.nx, s.p.ny / split_ra(s.p.ny), [&](auto l, auto r) -> hipError_t {
    constexpr int L = decltype(l)::value, RB = decltype(r)::value;
    using X = XS<T, L, RB>;
    if constexpr (!X::fits) {
      return hipErrorInvalidValue;
    } else {
      SMX_LAUNCH((k_xsplit<X>), dim3((unsigned)(s.p.ny / X::NC * s.p.nzh)), dim3(X::NT), 0, st, s);
      return hipGetLastError();
    }
  });
}
template <typename T>
hipError_t split_x_grp(const SplitArgs<T>* g, int nbox, const PParams<T>& p, hipStream_t st) {
  if (nbox < 1 || nbox > 65535) return hipErrorInvalidValue;
  return split_x_dispatch(p.nx, p.ny / split_ra(p.ny), [&](auto l, auto r) -> hipError_t {
    constexpr int L = decltype(l)::value, RB = decltype(r)::value;
    using X = XS<T, L, RB>;
    if constexpr (!X::fits) {
      return hipErrorInvalidValue;
    } else {
      SMX_LAUNCH((k_xsplit_grp<X>), dim3((unsigned)(p.ny / X::NC * p.nzh), (unsigned)nbox), dim3(X::NT), 0, st, g);
      return hipGetLastError();
    }
  });
}
template <typename T, typename TI>
hipError_t split_form_std(const cplx<TI>* in, cplx<T>* out, int64_t nrows, int ny, const cplx<T>* twy,
                          hipStream_t st) {
  if (nrows < 1) return hipErrorInvalidValue;
#define SMX_CASE(NY)                                                                                         \
  if (ny == NY) {                                                                                            \
    constexpr int RA = split_ra(NY), ROWS = 256 / RA;                                                        \
    SMX_LAUNCH((k_form_std<T, RA, NY / RA, TI>), dim3((unsigned)((nrows + ROWS - 1) / ROWS)), dim3(256), 0, st, in, \
               out, nrows, twy);                                                                             \
    return hipGetLastError();                                                                                \
  }
  SMX_FOR_EACH_SPLIT(SMX_CASE)
#undef SMX_CASE
  return hipErrorInvalidValue;
}
template <typename T>
hipError_t split_form(const cplx<T>* in, cplx<T>* out, int64_t nrows, int ny, const cplx<T>* twy, int dir,
                      const T* kmul, hipStream_t st) {
  if (nrows < 1 || (kmul != nullptr && dir != FORM_FROM_STD)) return hipErrorInvalidValue;
  if (dir == FORM_TO_STD) return split_form_std<T, T>(in, out, nrows, ny, twy, st);
  auto grid = [&](int rows) { return dim3((unsigned)((nrows + rows - 1) / rows)); };
#define SMX_CASE(NY)                                                                                              \
  if (ny == NY) {                                                                                                 \
    constexpr int RA = split_ra(NY), RB = NY / RA;                                                                \
    if (dir == FORM_FROM_STD)                                                                                     \
      SMX_LAUNCH((k_form_split<T, RA, RB>), grid(256 / RA), dim3(256), 0, st, in, out, nrows, twy, kmul);         \
    else if (dir == FORM_PERM_TO_STD)                                                                             \
      SMX_LAUNCH((k_form_perm<T, RA, RB, true>), grid(1024 / NY), dim3(256), 0, st, in, out, nrows);              \
    else                                                                                                          \
      SMX_LAUNCH((k_form_perm<T, RA, RB, false>), grid(1024 / NY), dim3(256), 0, st, in, out, nrows);             \
    return hipGetLastError();                                                                                     \
  }
  SMX_FOR_EACH_SPLIT(SMX_CASE)
#undef SMX_CASE
  return hipErrorInvalidValue;
}
#endif

#ifdef SMX_SPLIT_NEU_Z
template <typename T>
bool nsplit_z_fits(int nx, int ny, int nz) {
  const int ra = nsplit_ra(ny, nx);
  return ra != 0 && split_z_dispatch(nz, ra, [&](auto l, auto r) -> hipError_t {
           using Z = NZ<T, decltype(l)::value, decltype(r)::value>;
           return Z::fits && (ny / ra) % Z::NY2 == 0 ? hipSuccess : hipErrorInvalidValue;
         }) == hipSuccess;
}
template <typename T>
int nsplit_z_per_cu(int nx, int ny, int nz) {
  int n = 0;
  (void)split_z_dispatch(nz, nsplit_ra(ny, nx), [&](auto l, auto r) -> hipError_t {
    n = (int)(160 * 1024 / NZ<T, decltype(l)::value, decltype(r)::value>::BYTES);
    return hipSuccess;
  });
  return n;
}
template <typename T>
int nsplit_z_blocks(const PParams<T>& p) {
  const int ra = nsplit_ra(p.ny, p.nx);
  int n = 0;
  (void)split_z_dispatch(p.nz, ra, [&](auto l, auto r) -> hipError_t {
    n = p.nx * (p.ny / ra / NZ<T, decltype(l)::value, decltype(r)::value>::NY2);
    return hipSuccess;
  });
  return n;
}
template <typename T>
hipError_t nsplit_z(const SplitNeuArgs<T>& s, hipStream_t st) {
  return split_z_dispatch(s.p.nz, nsplit_ra(s.p.ny, s.p.nx), [&](auto l, auto r) -> hipError_t {
    using Z = NZ<T, decltype(l)::value, decltype(r)::value>;
    if constexpr (!Z::fits) {
      return hipErrorInvalidValue;
    } else {
      SMX_LAUNCH((k_nsplit_z<Z>), dim3((unsigned)(s.p.nx * (s.p.ny / Z::RA / Z::NY2))), dim3(Z::NT), 0, st, s);
      return hipGetLastError();
    }
  });
}
#endif

#ifdef SMX_SPLIT_NEU_X
template <typename T>
bool nsplit_x_fits(int nx, int ny) {
  const int ra = nsplit_ra(ny, nx);
  return ra != 0 && split_x_dispatch(nx, ny / ra, [&](auto l, auto r) -> hipError_t {
           using X = NX<T, decltype(l)::value, decltype(r)::value>;
           return X::fits && ny % X::NC == 0 ? hipSuccess : hipErrorInvalidValue;
         }) == hipSuccess;
}
template <typename T>
int nsplit_x_per_cu(int nx, int ny) {
  const int ra = nsplit_ra(ny, nx);
  int n = 0;
  if (ra != 0)
    (void)split_x_dispatch(nx, ny / ra, [&](auto l, auto r) -> hipError_t {
      n = (int)(160 * 1024 / NX<T, decltype(l)::value, decltype(r)::value>::BYTES);
      return hipSuccess;
    });
  return n;
}
template <typename T>
hipError_t nsplit_x(const SplitNeuArgs<T>& s, hipStream_t st) {
  return split_x_dispatch(s.p.nx, s.p.ny / nsplit_ra(s.p.ny, s.p.nx), [&](auto l, auto r) -> hipError_t {
    using X = NX<T, decltype(l)::value, decltype(r)::value>;
    if constexpr (!X::fits) {
      return hipErrorInvalidValue;
    } else {
      SMX_LAUNCH((k_nsplit_x<X>), dim3((unsigned)(s.p.ny / X::NC * (s.p.nz / 2))), dim3(X::NT), 0, st, s);
      return hipGetLastError();
    }
  });
}
#endif

#if defined(SMX_SPLIT_NEU_REAL) || defined(SMX_SPLIT_SURF)
// FP64 tiles also of the grids whose FP32 step fits: one y2 where two do not.
template <int L, int RA>
using NZReal = NZ<double, L, RA, NZ<double, L, RA>::fits ? nsplit_ny2<double>(L, RA) : 1>;
#endif

#ifdef SMX_SPLIT_SURF
template <typename TI>
hipError_t split_scan_surf(const cplx<TI>* a, const PParams<double>& p, const SplitScan& s, hipStream_t st) {
  return split_z_dispatch(p.nz, split_ra(p.ny), [&](auto l, auto r) -> hipError_t {
    using Z = ZS<double, decltype(l)::value, decltype(r)::value>;
    if constexpr (!split_scan_fits<Z, 2>()) {
      return hipErrorNotSupported;
    } else {
      SMX_LAUNCH((k_zsplit_scan<Z, TI>), dim3((unsigned)(p.nx * (p.ny / Z::RA / Z::NY2))), dim3(Z::NT), 0, st, a, p, s);
      return hipGetLastError();
    }
  });
}
template <typename TI>
hipError_t nsplit_scan_surf(const cplx<TI>* a, const PParams<double>& p, const cplx<double>* qtz, const SplitScan& s,
                            hipStream_t st) {
  return split_z_dispatch(p.nz, nsplit_ra(p.ny, p.nx), [&](auto l, auto r) -> hipError_t {
    using Z = NZReal<decltype(l)::value, decltype(r)::value>;
    if constexpr (!split_scan_fits<Z, 4>()) {
      return hipErrorNotSupported;
    } else {
      SMX_LAUNCH((k_nsplit_scan<Z, TI>), dim3((unsigned)(p.nx * (p.ny / Z::RA / Z::NY2))), dim3(Z::NT), 0, st, a, p, qtz,
                 s);
      return hipGetLastError();
    }
  });
}
#endif

#ifdef SMX_SPLIT_NEU_REAL
bool nsplit_real_fits(int nx, int ny, int nz) {
  const int ra = nsplit_ra(ny, nx);
  return ra != 0 && split_z_dispatch(nz, ra, [&](auto l, auto r) -> hipError_t {
           using Z = NZReal<decltype(l)::value, decltype(r)::value>;
           return Z::fits && (ny / ra) % Z::NY2 == 0 ? hipSuccess : hipErrorInvalidValue;
         }) == hipSuccess;
}
template <typename TI>
hipError_t nsplit_real(const cplx<TI>* a, double* out, const PParams<double>& p, const cplx<double>* qtz,
                       hipStream_t st) {
  return split_z_dispatch(p.nz, nsplit_ra(p.ny, p.nx), [&](auto l, auto r) -> hipError_t {
    using Z = NZReal<decltype(l)::value, decltype(r)::value>;
    if constexpr (!Z::fits) {
      return hipErrorInvalidValue;
    } else {
      SMX_LAUNCH((k_nsplit_real<Z, TI>), dim3((unsigned)(p.nx * (p.ny / Z::RA / Z::NY2))), dim3(Z::NT), 0, st, a, out, p,
                 qtz);
      return hipGetLastError();
    }
  });
}
template <typename TI, typename TO, int RA, int RB>
static hipError_t nsplit_form_dir(const TI* in, TO* out, int nx, int nz, const cplx<double>* twy,
                                  const cplx<double>* qty, int dir, hipStream_t st) {
  constexpr int ROWS = 128 / RA;
  const dim3 grid((unsigned)((nx * (nz / 2) + ROWS - 1) / ROWS));
  if (dir == FORM_TO_STD) {
    SMX_LAUNCH((k_nform_std<TI, TO, RA, RB>), grid, dim3(128), 0, st, in, out, nx, nz, twy, qty);
  } else if constexpr (std::is_same_v<TI, TO>) {
    if (dir == FORM_FROM_STD)
      SMX_LAUNCH((k_nform_split<TI, RA, RB>), grid, dim3(128), 0, st, in, out, nx, nz, twy, qty);
    else if (dir == FORM_PERM_TO_STD)
      SMX_LAUNCH((k_nform_perm<TI, RA, RB, true>), grid, dim3(128), 0, st, in, out, nx, nz);
    else
      SMX_LAUNCH((k_nform_perm<TI, RA, RB, false>), grid, dim3(128), 0, st, in, out, nx, nz);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
template <typename TI, typename TO>
hipError_t nsplit_form(const TI* in, TO* out, int nx, int ny, int nz, const cplx<double>* twy, const cplx<double>* qty,
                       int dir, hipStream_t st) {
  const int ra = nsplit_ra(ny, nx);
#define SMX_CASE(NY)                                                                                              \
  if (ny == NY) {                                                                                                 \
    constexpr int R0 = nsplit_ra(NY, 1), R3 = nsplit_ra(NY, 3);                                                   \
    return ra == R0 ? nsplit_form_dir<TI, TO, R0, NY / R0>(in, out, nx, nz, twy, qty, dir, st)                    \
                    : nsplit_form_dir<TI, TO, R3, NY / R3>(in, out, nx, nz, twy, qty, dir, st);                   \
  }
  SMX_FOR_EACH_SPLIT(SMX_CASE)
#undef SMX_CASE
  return hipErrorInvalidValue;
}
#endif

}  // namespace smx
