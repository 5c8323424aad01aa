// smx_split_adv.h -- the advected periodic step (smx_advect.h) in four launches, with the y transforms
// divided between the z and the x kernels (smx_split.h):
//   k_zsplit_force  A, Ax, Ay, As -> S0, S1, S2       S = f grad psi
//   k_xsplit_stokes S -> U                            U = s CM1 (S - CM2 (k.S)), in place
//   k_zsplit_advnl  U0..2, A, Ax, Ay -> N             N = N(psi) - U.grad psi
//   k_xsplit_adv    N, R -> R, A, Ax, Ay, As          CNAB2; psi, d_x psi, d_y psi, psiSH
// S0, U0 and N take As's array, as in the fifteen launches.  27 moves of a stage array instead of 48: the
// eleven y passes go, and d_y psi is formed in the x kernel, which has k_y at hand, so it is a fifth
// carried array.
// 256^3 FP32: 148 + 170 + 198 + 122 us against 680 in fifteen launches; FP64 1210 against 1410; 96 x 64 x
// 128 FP64, where the launches and their gaps are the larger part, 97 against 138 us a step.  Moves alone
// would take 262 us of the 638: the z kernels are bound by their transforms (seven inverse and one forward
// in k_zsplit_advnl, each with two or three trips through LDS between barriers, and two blocks a CU to
// cover them), k_xsplit_stokes by the 157 to 170 registers of three fields a thread (one block of 512
// threads a CU).
#pragma once
#include "smx_advect.h"
#include "smx_split.h"

namespace smx {

template <typename T>
struct SplitAdvArgs {
  cplx<T>*a, *ax, *ay, *as, *s1, *s2;  // stage arrays, split form
  cplx<T>* r;                          // carry, split form
  const cplx<T>* twy;
  AParams<T> ap;
};

// Tiles: those of k_zsplit and k_xsplit (with the k_z table), x blocks of at most 512 threads (a
// thread of the Stokes kernel holds three fields, 128 registers or more).
template <typename Z>
constexpr bool zsa_fits() {
  return Z::fits && (size_t)(Z::LDS + Z::L) * sizeof(cplx<typename Z::T>) + Z::RED * 8 +
                            Z::NZH * sizeof(typename Z::T) <= 160 * 1024;
}
template <typename X>
constexpr bool xsa_fits() {
  return X::fits && X::NT <= 512;
}

#define SMX_ZSA_SETUP(ARGS, NPROJ)                                                               \
  using T = typename Z::T;                                                                      \
  constexpr int E = Z::E, L = Z::L;                                                             \
  __shared__ cplx<T> F[Z::LDS];                                                                 \
  __shared__ cplx<T> TW[L];                                                                     \
  __shared__ T KZ[Z::NZH];                                                                      \
  const PParams<T>& p = ARGS.ap.p;                                                              \
  const int tid = threadIdx.x, q = tid % Z::NPR, tc = tid / Z::NPR;                             \
  const int bz = (int)blockIdx.x - (NPROJ);                                                     \
  if (bz < 0) {                                                                                 \
    split_project(ARGS.r, p, Z::RA, blockIdx.x, NPROJ, tid, Z::NT);                             \
    return;                                                                                     \
  }                                                                                             \
  const cplx<T>* twl = tw_lds<L, Z::NT>(TW, p.twz, tid);                                        \
  for (int i = tid; i < Z::NZH; i += Z::NT) KZ[i] = p.kz[i];                                    \
  const int rb = p.ny / Z::RA;                                                                  \
  int x, yg;                                                                                    \
  zs_tile(bz, rb / Z::NY2, x, yg);                                                              \
  const uint32_t rowb = (uint32_t)p.nxy * (uint32_t)sizeof(cplx<T>);                            \
  const int64_t ofs = (int64_t)x * p.ny + split_pos(0, yg * Z::NY2, rb);                               \
  __syncthreads();  /* KZ */

// Force S = f grad psi (pf3d.cpp:417-425), f = psiSH or mu = psiSH - eps psi - N(psi).
template <typename Z>
__global__ __launch_bounds__(Z::NT) void k_zsplit_force(SplitAdvArgs<typename Z::T> s, int nproj) {
  SMX_ZSA_SETUP(s, nproj)
  // lane indices made again for each transform: its address arithmetic then stays where it is used
  // instead of being kept in registers across all of them
  auto inverse = [&](const cplx<T>* in, const T* kzm, cplx<T>* v) {
    __syncthreads();  // the tile's last reads are done
    int ti = tid, qi = q, ci = tc;
    asm volatile("" : "+v"(ti), "+v"(qi), "+v"(ci));
    zs_inverse<Z>(in + ofs, rowb, rb, F, twl, ti, qi, ci, v, kzm);
  };
  cplx<T> f[E], v[E];
  inverse(s.as, nullptr, f);
  if (s.ap.force == F_MU) {
    inverse(s.a, nullptr, v);
#pragma unroll
    for (int e = 0; e < E; ++e)
      f[e] = mk(f[e].x - p.eps * v[e].x - nonlin(p, v[e].x), f[e].y - p.eps * v[e].y - nonlin(p, v[e].y));
  }
#pragma unroll 1
  for (int c = 0; c < 3; ++c) {
    inverse(c == 0 ? s.ax : (c == 1 ? s.ay : s.a), c == 2 ? KZ : nullptr, v);
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = mk(f[e].x * v[e].x, f[e].y * v[e].y);
    int ti = tid, qi = q, ci = tc;
    asm volatile("" : "+v"(ti), "+v"(qi), "+v"(ci));
    zs_forward<Z>(v, (c == 0 ? s.as : (c == 1 ? s.s1 : s.s2)) + ofs, rowb, rb, F, twl, ti, qi, ci);
  }
}

// N = N(psi) - U.grad psi [+ mid-plane penalty] (pf3d.cpp:455-465, pf3dMorph.cpp:572-590).
template <typename Z>
__global__ __launch_bounds__(Z::NT) void k_zsplit_advnl(SplitAdvArgs<typename Z::T> s) {
  __shared__ double red[Z::RED];
  SMX_ZSA_SETUP(s, 0)
  constexpr int RP = fwd_first<L, Z::V>();
  auto inverse = [&](const cplx<T>* in, const T* kzm, cplx<T>* v) {  // as in k_zsplit_force
    __syncthreads();
    int ti = tid, qi = q, ci = tc;
    asm volatile("" : "+v"(ti), "+v"(qi), "+v"(ci));
    zs_inverse<Z>(in + ofs, rowb, rb, F, twl, ti, qi, ci, v, kzm);
  };
  cplx<T> v[E], u[E], nacc[E];
  inverse(s.a, nullptr, v);
  const bool pen = p.mid > 0 && p.mid < L - 1;
  if (pen) {
    __syncthreads();
    Tile<T, L, E, Z::FP>::template store<RP>(v, F, q, tc);
    __syncthreads();
  }
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int n = Tile<T, L, E, Z::FP>::template pos_in<RP>(tc, e);
    T a = nonlin(p, v[e].x), b = nonlin(p, v[e].y);
    if (pen && n == p.mid) {
      const cplx<T> lo = F[(n - 1) * Z::FP + q], hi = F[(n + 1) * Z::FP + q];
      a += p.pen * (lo.x - (T)2 * v[e].x + hi.x);
      b += p.pen * (lo.y - (T)2 * v[e].y + hi.y);
    }
    nacc[e] = mk(a, b);
  }
#pragma unroll 1
  for (int c = 0; c < 3; ++c) {
    inverse(c == 0 ? s.as : (c == 1 ? s.s1 : s.s2), nullptr, u);
    inverse(c == 0 ? s.ax : (c == 1 ? s.ay : s.a), c == 2 ? KZ : nullptr, v);
#pragma unroll
    for (int e = 0; e < E; ++e) nacc[e] = mk(nacc[e].x - u[e].x * v[e].x, nacc[e].y - u[e].y * v[e].y);
  }
  if (p.partial != nullptr) zs_partial<T, E, Z::NT>(nacc, red, tid);
  zs_forward<Z>(nacc, s.as + ofs, rowb, rb, F, twl, tid, q, tc);  // its barriers order red[]
  if (p.partial != nullptr && tid == 0) {
    double t = 0.0;
    for (int w = 0; w < Z::RED; ++w) t += red[w];
    p.partial[bz] = t;
  }
}
#undef SMX_ZSA_SETUP

// AGAIN: lane indices made again for each transform, as in k_zsplit_force, for the kernels that spill otherwise, or
// whose registers keep a second block off the CU (it costs the others 3 to 5%).  Stokes in FP64 on lines of 384, and
// of 256 with 16 y2: 384 x 192 x 256 595 -> 505 us, 384 x 96 x 64 126 -> 109, 256^3 298 -> 274; the update in FP32 on
// lines of 384 (k_xsplit_adv): 384 x 192 x 256 216 -> 164 us, 384 x 96 x 512 251 -> 204.
#define SMX_XSA_SETUP(ARGS, AGAIN)                                                                 \
  using T = typename X::T;                                                                        \
  constexpr int L = X::L, RB = X::RB, NC = X::NC, V = X::V;                                       \
  constexpr int E = X::E, NT = X::NT, NCP = X::NCP, NK = X::NK;                                   \
  constexpr uint32_t CB = sizeof(cplx<T>);                                                        \
  using AD = typename X::AD;                                                                      \
  using TL = Tile<T, L, E, NCP>;                                                                  \
  __shared__ cplx<T> S[L * NCP];                                                                  \
  __shared__ cplx<T> TW[L];                                                                       \
  __shared__ T KX[L];                                                                             \
  const PParams<T>& p = ARGS.ap.p;                                                                \
  const int tid = threadIdx.x, col = tid % NC, tc = tid / NC;                                     \
  int bx, kz;                                                                                     \
  xs_tile<X>(blockIdx.x, p.ny / NC, p.nzh, bx, kz);                                               \
  const cplx<T>* twl = tw_lds<L, NT>(TW, p.twx, tid);                                             \
  for (int i = tid; i < L; i += NT) KX[i] = p.kx[i];                                              \
  const cplx<T> tw = ARGS.twy[(bx * NK + col / RB) * (col % RB)];  /* w_ny^{y2 k1} */             \
  const int ky = bx * NK + col / RB + p.ny / RB * (col % RB);                                     \
  const int64_t plane = (int64_t)kz * p.nxy;                                                      \
  const uint32_t rowb = (uint32_t)p.ny * CB;                                                      \
  const uint32_t aofs = (uint32_t)split_pos(bx * NK + col / RB, col % RB, RB) * CB;                \
  const T kyv = p.ky[ky], kzv = p.kz[kz];                                                         \
  auto forward = [&](cplx<T>* w) {                                                                \
    int ti = tid, ci = col, cc = tc;                                                              \
    if constexpr (AGAIN) asm volatile("" : "+v"(ti), "+v"(ci), "+v"(cc));                         \
    _Pragma("unroll") for (int e = 0; e < E; ++e) w[e] = cmul(w[e], tw);                          \
    RowFFT<true, T, L, E, AD, -1, typename PlanV<L, V>::Fwd>::run(w, S, ci, cc, twl,              \
                                                                  [&]() { XRow<X, -1>::run(S, ti); }); \
  };                                                                                              \
  auto inverse = [&](cplx<T>* w) {                                                                \
    int ti = tid, ci = col, cc = tc;                                                              \
    if constexpr (AGAIN) asm volatile("" : "+v"(ti), "+v"(ci), "+v"(cc));                         \
    RowFFT<true, T, L, E, AD, +1, typename PlanV<L, V>::Inv>::run(w, S, ci, cc, twl,              \
                                                                  [&]() { XRow<X, +1>::run(S, ti); }); \
    _Pragma("unroll") for (int e = 0; e < E; ++e) w[e] = cmul(w[e], conjg(tw));                   \
  };

// Stokes projection in full k-space (pf3d.cpp:433-447), U(k = 0) = 0.
template <typename X>
__global__ __launch_bounds__(X::NT) void k_xsplit_stokes(SplitAdvArgs<typename X::T> s) {
  SMX_XSA_SETUP(s, (sizeof(typename X::T) == 8 && (X::L > 256 || (X::L == 256 && X::RB == 16))))
  cplx<T>* arr[3] = {s.as + plane, s.s1 + plane, s.s2 + plane};
  cplx<T> v[3][E];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
#pragma unroll
    for (int e = 0; e < E; ++e)
      v[c][e] = ld_off<cplx<T>>(arr[c], (uint32_t)TL::template pos_in<fwd_first<L, V>()>(tc, e) * rowb + aofs);
    forward(v[c]);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int kxi = TL::template pos_in<fwd_last<L, V>()>(tc, e);
    const T kxv = KX[kxi];
    const T k2 = kxv * kxv + kyv * kyv + kzv * kzv;
    const cplx<T> a0 = v[0][e], a1 = v[1][e], a2 = v[2][e];
    cplx<T> u0 = mk<T>(0, 0), u1 = mk<T>(0, 0), u2 = mk<T>(0, 0);
    if (!(kxi == 0 && ky == 0 && kz == 0)) {  // CM1[0] = CM2[0] = 0 (pf3d.cpp:219-222)
      const cplx<T> dot = mk(kxv * a0.x + kyv * a1.x + kzv * a2.x, kxv * a0.y + kyv * a1.y + kzv * a2.y);
      const T ik2 = recip(k2);
      const T cm1 = p.scale * s.ap.cm * ik2;
      const T c2x = kxv * ik2, c2y = kyv * ik2, c2z = kzv * ik2;
      u0 = mk(cm1 * (a0.x - c2x * dot.x), cm1 * (a0.y - c2x * dot.y));
      u1 = mk(cm1 * (a1.x - c2y * dot.x), cm1 * (a1.y - c2y * dot.y));
      u2 = mk(cm1 * (a2.x - c2z * dot.x), cm1 * (a2.y - c2z * dot.y));
    }
    v[0][e] = u0;
    v[1][e] = u1;
    v[2][e] = u2;
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    inverse(v[c]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < E; ++e)
      st_off(arr[c], (uint32_t)TL::template pos_in<inv_last<L, V>()>(tc, e) * rowb + aofs, v[c][e]);
  }
}

// CNAB2 update (as k_xsplit) with four inverse outputs.  AGAIN in FP32 on lines of 384 with more blocks than CUs
// (132 blocks, 384 x 64 x 64: a step 92.4 us without, 95.1).
template <typename X, bool AGAIN>
__global__ __launch_bounds__(X::NT) void k_xsplit_adv(SplitAdvArgs<typename X::T> s) {
  SMX_XSA_SETUP(s, AGAIN)
  const uint32_t cofs = (uint32_t)(bx * NC + col) * CB;
  cplx<T>* rb = s.r + plane;
  cplx<T> v[E], ps[E];
#pragma unroll
  for (int e = 0; e < E; ++e)
    v[e] = ld_off<cplx<T>>(s.as + plane, (uint32_t)TL::template pos_in<fwd_first<L, V>()>(tc, e) * rowb + aofs);
  double nsum = 0.0;
  const bool owner0 = (p.partial != nullptr) && kz == 0 && bx == 0;
  if (owner0) nsum = xs_partial_sum<X>(p, S, tid);
  forward(v);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int kxi = TL::template pos_in<fwd_last<L, V>()>(tc, e);
    const uint32_t o = (uint32_t)kxi * rowb + cofs;
    const T kxv = KX[kxi];
    const T aLin = p.eps - op_sh(p, kxv * kxv + kyv * kyv + kzv * kzv);
    const T C1 = (T)1 + p.dtd2 * aLin, C2 = (T)1 - p.dtd2 * aLin;
    const cplx<T> nn = p.scale * v[e];
    const cplx<T> r = ld_off<cplx<T>>(rb, o);  // pf3d.cpp:476-478 with R = C1 psi - dt/2 N_past
    const T ic2 = recip(C2);
    cplx<T> ps1 = mk(ic2 * (r.x + (T)3 * p.dtd2 * nn.x), ic2 * (r.y + (T)3 * p.dtd2 * nn.y));
    cplx<T> rn = mk(C1 * ps1.x - p.dtd2 * nn.x, C1 * ps1.y - p.dtd2 * nn.y);
    if (owner0 && tid == 0 && kxi == 0) {
      const double dd = p.m_dtd2, n0 = p.m_scale * nsum;
      const double ps0 = (p.mean_state[0] + 3.0 * dd * n0) / p.m_c2;
      p.mean_state[0] = p.m_c1 * ps0 - dd * n0;
      p.mean_state[1] = ps0;
      ps1 = mk((T)ps0, (T)0);
      rn = mk((T)p.mean_state[0], (T)0);
    }
    st_off(rb, o, rn);
    ps[e] = ps1;
  }
#pragma unroll 1
  for (int o = 0; o < 4; ++o) {
    cplx<T>* dst = (o == 0 ? s.a : (o == 1 ? s.ax : (o == 2 ? s.ay : s.as))) + plane;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const T kxv = KX[TL::template pos_in<fwd_last<L, V>()>(tc, e)];
      if (o == 0) v[e] = ps[e];
      else if (o == 1) v[e] = mk(-kxv * ps[e].y, kxv * ps[e].x);  // i kx psi_hat (pf3d.cpp:404)
      else if (o == 2) v[e] = mk(-kyv * ps[e].y, kyv * ps[e].x);  // i ky psi_hat (:405)
      else v[e] = op_sh(p, kxv * kxv + kyv * kyv + kzv * kzv) * ps[e];  // opSH psi_hat (:407)
    }
    inverse(v);
#pragma unroll
    for (int e = 0; e < E; ++e)
      st_off(dst, (uint32_t)TL::template pos_in<inv_last<L, V>()>(tc, e) * rowb + aofs, v[e]);
  }
}
#undef SMX_XSA_SETUP

}  // namespace smx
