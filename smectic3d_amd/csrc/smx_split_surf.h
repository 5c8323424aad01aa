// smx_split_surf.h -- surfTrack's psi, column scan and z derivative from a split-form state in one kernel:
//   k_zsplit_scan  periodic (smx_split.h):    psi, the crossings and psi_z at them
//   k_nsplit_scan  Neumann (smx_split_neu.h): psi, the crossings and psi_zz at them
// The inverse half of the z kernel, then what k_zinv_scan and k_dct_zinv_scan (smx_surf.h) do with their tile:
// psi's rows to memory, one wave per column for the scan, and the derivative at each column's evaluation index
// from the lines' spectra, which stay in the registers of the items that the inverse half made them in.  In
// place of the standard form's y inverse and scan, two more moves of a stage array in FP64: 256 x 256 x 384 164
// us from FP32 (71 + 124), 256^3 FP64 79 (45 + 73).  The Neumann one is bound by the work of one block a CU
// (117 KB): the inverse half alone takes 93 us, psi's rows 40, the scan 15, the sums 15; two blocks of half the
// tile were no faster.
#pragma once
#include "smx_split.h"
#include "smx_split_neu.h"

namespace smx {

// The scan of a tile F of NP column pairs (in x and y, z at its index, an odd pitch: lanes run along z), one wave
// per pair: from the bottom (DOWN: from the top), armed above `arm`, the first psi < 0; its evaluation index is
// that point or the one before it, whichever is nearer to zero.  put(q, half, crossing, evaluation index) by one
// lane per column; -1 without a crossing.
template <int L, int NP, int NT, int FP, bool DOWN, typename Put>
__device__ __forceinline__ void split_scan(const cplx<double>* F, double arm, int tid, Put&& put) {
  constexpr int CH = (L + 63) / 64;
  const int lane = tid & 63;
  auto at = [&](int i) { return DOWN ? L - 1 - i : i; };  // z of the scan's i-th point
  for (int q = tid >> 6; q < NP; q += NT / 64) {
    cplx<double> w[CH];
#pragma unroll
    for (int ch = 0; ch < CH; ++ch) {
      const int i = ch * 64 + lane;
      w[ch] = i < L ? F[at(i) * FP + q] : mk<double>(0, 0);
    }
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      bool armed = false;
      int f = -1;
#pragma unroll
      for (int ch = 0; ch < CH; ++ch) {  // a lane past L holds 0 and takes no part
        const double val = half ? w[ch].y : w[ch].x;
        const uint64_t am = __ballot(ch * 64 + lane < L && val > arm);
        uint64_t neg = __ballot(val < 0.0);
        if (f < 0) {
          if (!armed && am) {
            neg &= ~0ull << (__ffsll((unsigned long long)am) - 1);
            armed = true;
          }
          if (armed && neg) f = ch * 64 + __ffsll((unsigned long long)neg) - 1;
        }
      }
      if (lane == 0) {
        auto P = [&](int i) {
          const cplx<double> g = F[at(i) * FP + q];
          return fabs(half ? g.y : g.x);
        };
        put(q, half, f < 0 ? -1 : at(f), f < 0 ? -1 : at(f > 0 && P(f) > P(f - 1) ? f - 1 : f));
      }
    }
  }
}

// Sums of acc[k] over the threads of equal tid % G, into out(k, g) by one thread each, in a fixed order: H values
// by a thread, then the partial sums of a line.  R: (H + 1) NT doubles that nothing else uses.
template <int H, int G, int NT, typename Out>
__device__ __forceinline__ void split_line_sums(const double* acc, double* R, int tid, Out&& out) {
  constexpr int NL = G * H, PT = NT / NL, PER = NT / G / PT;  // lines, threads of a line, values of a thread
  static_assert(NT % NL == 0 && PER * PT * G == NT, "whole threads");
  double* R1 = R + H * NT;
#pragma unroll
  for (int k = 0; k < H; ++k) R[k * NT + tid] = acc[k];
  __syncthreads();
  const int i = tid / PT, u = tid - i * PT, k = i % H, g = i / H;
  double s = 0.0;
#pragma unroll
  for (int e = 0; e < PER; ++e) s += R[k * NT + (e * PT + u) * G + g];
  R1[tid] = s;
  __syncthreads();
  if (u == 0) {
#pragma unroll
    for (int w = 1; w < PT; ++w) s += R1[tid + w];
    out(k, g, s);
  }
}

// Whether a z tile takes the scan: whole waves, and room in the tile for the trigonometric table and the sums.
template <typename Z, int TRIG>
constexpr bool split_scan_fits() {
  return Z::fits && Z::NT % 64 == 0 && Z::NT % (Z::RA * Z::NY2) == 0 &&
         2 * Z::SLDS >= TRIG * Z::L + (Z::H + 1) * Z::NT &&
         (size_t)(Z::SLDS + Z::L) * sizeof(cplx<double>) + 2 * Z::NPR * sizeof(int) <= 160 * 1024;
}

// trig: k_surf_tables' table (periodic: 2 nz values, Neumann: 4 nz).  dz: ns parts of nxy, the sum in part 0
// and zeros in the others.
struct SplitScan {
  double* psi;
  const double* trig;
  double arm;
  int *kc, *ke;
  int ns;
  double* dz;
};

// psi_z at n: y = sum_{m=0}^{nz/2} w_m Re(i k_z X_m e^{2 pi i m n / nz}), w_0 = w_{nz/2} = 1, else 2; only the
// real parts of X_0 and X_{nz/2} enter, as in psi itself.
template <typename Z, typename TI>
__global__ __launch_bounds__(Z::NT) void k_zsplit_scan(const cplx<TI>* a, PParams<double> p, SplitScan s) {
  constexpr int L = Z::L, RA = Z::RA, NC = 2 * Z::NPR, G = Z::P * Z::NY2, SP = Z::SP;
  __shared__ cplx<double> F[Z::SLDS];
  __shared__ cplx<double> TW[L];
  __shared__ int KE[NC];
  const int tid = threadIdx.x, q = tid % Z::NPR, tc = tid / Z::NPR;
  const int rb = p.ny / RA;
  int x, yg;
  zs_tile(blockIdx.x, rb / Z::NY2, x, yg);
  cplx<double> v[Z::E], w[Z::IPT][Z::H];
  zs_inverse_w<Z, TI>(a + (int64_t)x * p.ny + split_pos(0, yg * Z::NY2, rb),
                      (uint32_t)p.nxy * (uint32_t)sizeof(cplx<TI>), rb, F, TW, tid, q, tc, v, w,
                      (const double*)nullptr, p.twz);
  __syncthreads();
  Tile<double, L, Z::E, SP>::template store<inv_last<L, Z::V>()>(v, F, q, tc);
  __syncthreads();
  const int64_t c0 = (int64_t)x * p.ny + yg * Z::NY2;  // column of y1 = 0, c = 0
  for (int i = tid; i < Z::NPR * L; i += Z::NT) {      // as k_zsplit_real
    const int qq = i / L, n = i - qq * L;
    const cplx<double> g = F[n * SP + qq];
    double* row = s.psi + (c0 + 2 * (qq / Z::NY2) * rb + qq % Z::NY2) * L;
    row[n] = g.x;
    row[(int64_t)rb * L + n] = g.y;
  }
  split_scan<L, Z::NPR, Z::NT, SP, false>(F, s.arm, tid, [&](int qq, int half, int kc, int ke) {
    const int64_t col = c0 + (2 * (qq / Z::NY2) + half) * rb + qq % Z::NY2;
    s.kc[col] = kc;
    s.ke[col] = ke;
    KE[2 * qq + half] = ke;
  });
  __syncthreads();  // KE, and every read of the tile is done
  double* TR = reinterpret_cast<double*>(F);
  for (int i = tid; i < 2 * L; i += Z::NT) TR[i] = s.trig[i];
  const int lo = tid % Z::P, cy = tid / Z::P % Z::NY2;  // of all the thread's items: NT is a multiple of G
  int n[Z::H];
  double acc[Z::H];
#pragma unroll
  for (int k = 0; k < Z::H; ++k) {
    n[k] = KE[2 * ((lo * Z::HC + k / 2) * Z::NY2 + cy) + (k & 1)];
    acc[k] = 0.0;
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < Z::IPT; ++it) {
    const int i = tid + it * Z::NT, m = i / G;
    if (i < Z::ITEMS) {
      const double im = (m == 0 || m == L / 2) ? 0.0 : 1.0, wk = ((m == 0 || m == L / 2) ? 1.0 : 2.0) * p.kz[m];
#pragma unroll
      for (int k = 0; k < Z::H; ++k) {
        const uint32_t j = n[k] >= 0 ? ((uint32_t)m * (uint32_t)n[k]) % (uint32_t)L : 0u;
        acc[k] -= wk * (im * w[it][k].y * TR[j] + w[it][k].x * TR[L + j]);
      }
    }
  }
  split_line_sums<Z::H, G, Z::NT>(acc, TR + 2 * L, tid, [&](int k, int g, double sum) {
    const int64_t col = c0 + (g % Z::P * Z::H + k) * rb + g / Z::P;  // y1 = lo H + k
    s.dz[col] = sum;
    for (int i = 1; i < s.ns; ++i) s.dz[i * p.nxy + col] = 0.0;
  });
}

// psi_zz at n: y = sum_k w_k (-k_z^2) x_k cos(pi k (2n+1) / 2nz), w_0 = 1, else 2.  The cosine of the partner
// nz - k is (-1)^n sin(pi k (2n+1) / 2nz), a quarter of the table's period away.
template <typename Z, typename TI>
__global__ __launch_bounds__(Z::NT) void k_nsplit_scan(const cplx<TI>* a, PParams<double> p,
                                                       const cplx<double>* __restrict__ qtz, SplitScan s) {
  constexpr int L = Z::L, NC = 2 * Z::NPR, G = Z::P * Z::NY2, SP = Z::SP;
  __shared__ cplx<double> F[Z::SLDS];
  __shared__ cplx<double> TW[L];
  __shared__ int KE[NC];
  const int tid = threadIdx.x, q = tid % Z::NPR, tc = tid / Z::NPR;
  const int rb = p.ny / Z::RA;
  int x, yg;
  zs_tile(blockIdx.x, rb / Z::NY2, x, yg);
  cplx<double> v[Z::E], qw[Z::IPT][2], w[Z::IPT][Z::H];
  nz_twiddles<Z>(qtz, tid, qw);
  nz_inverse_w<Z, TI>(a + (int64_t)x * p.ny + split_pos(0, yg * Z::NY2, rb),
                      (uint32_t)p.nxy * (uint32_t)sizeof(cplx<TI>), rb, F, TW, p.twz, qw, tid, q, tc, v, w);
  __syncthreads();
#pragma unroll
  for (int e = 0; e < Z::E; ++e)
    F[mk_src(Tile<double, L, Z::E, Z::HP>::template pos_in<inv_last<L, Z::V>()>(tc, e), L) * SP + q] = v[e];
  __syncthreads();
  auto column = [&](int y1, int c) { return (int64_t)x * p.ny + mk_src(y1 * rb + yg * Z::NY2 + c, p.ny); };
  for (int i = tid; i < Z::NPR * L; i += Z::NT) {  // as k_nsplit_real
    const int qq = i / L, n = i - qq * L;
    const int c = qq % Z::NY2, h = qq / Z::NY2 % Z::HC, lo = qq / Z::NY2 / Z::HC, ya = 2 * h * Z::P + lo;
    const cplx<double> g = F[n * SP + qq];
    s.psi[column(ya, c) * L + n] = g.x;
    s.psi[column(ya + Z::P, c) * L + n] = g.y;
  }
  split_scan<L, Z::NPR, Z::NT, SP, true>(F, s.arm, tid, [&](int qq, int half, int kc, int ke) {
    const int h = qq / Z::NY2 % Z::HC, lo = qq / Z::NY2 / Z::HC;
    const int64_t col = column((2 * h + half) * Z::P + lo, qq % Z::NY2);
    s.kc[col] = kc;
    s.ke[col] = ke;
    KE[2 * qq + half] = ke;
  });
  __syncthreads();  // KE, and every read of the tile is done
  double* TR = reinterpret_cast<double*>(F);
  for (int i = tid; i < 4 * L; i += Z::NT) TR[i] = s.trig[i];
  const int lo = tid % Z::P, cy = tid / Z::P % Z::NY2;
  uint32_t st[Z::H];
  double acc[Z::H];
#pragma unroll
  for (int k = 0; k < Z::H; ++k) {
    const int n = KE[2 * ((lo * Z::HC + k / 2) * Z::NY2 + cy) + (k & 1)];
    st[k] = n >= 0 ? 2 * n + 1 : 0;
    acc[k] = 0.0;
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < Z::IPT; ++it) {
    const int i = tid + it * Z::NT, j = i / G, jp = j == 0 ? L / 2 : L - j;
    if (i < Z::ITEMS) {
      const double ka = p.kz[j], kb = p.kz[jp], wa = (j == 0 ? -1.0 : -2.0) * ka * ka, wb = -2.0 * kb * kb;
#pragma unroll
      for (int k = 0; k < Z::H; ++k) {
        const uint32_t ia = (uint32_t)j * st[k] % (4u * L);
        const uint32_t ib = j == 0 ? (L / 2) * (st[k] & 7) : ia >= L ? ia - L : ia + 3 * L;
        const double sb = j != 0 && (st[k] & 2) ? -wb : wb;
        acc[k] += wa * w[it][k].x * TR[ia] + sb * w[it][k].y * TR[ib];
      }
    }
  }
  split_line_sums<Z::H, G, Z::NT>(acc, TR + 4 * L, tid, [&](int k, int g, double sum) {
    const int64_t col = column(k * Z::P + g % Z::P, g / Z::P);
    s.dz[col] = sum;
    for (int i = 1; i < s.ns; ++i) s.dz[i * p.nxy + col] = 0.0;
  });
}

}  // namespace smx
