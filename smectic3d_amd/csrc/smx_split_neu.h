// smx_split_neu.h -- the plain Neumann step (smx_neumann.h) in two launches, with the y transform divided
// between the z and the x kernel as in smx_split.h.
//
// The cosine transforms are real-linear, so two planes kz travel as the real and the imaginary part of one
// complex plane through x and y, where no untangling is needed: planes j and nz - j (0 and nz/2 for j = 0).
// Along y, DCT-II of such a line is FFT of the reordered line, then X[k] = w_k V[k] + conj(w_k) V[ny-k], and
// DCT-III the inverse steps; the FFT's radix RA (over y1 of m = y1 RB + y2, src(m) the point) is the z
// kernel's, the rest the x kernel's:
//   k_nsplit_z  radix RA over k1, DCT-III z, N(psi), DCT-II z, radix RA over y1
//   k_nsplit_x  forward x FFT with radix RB over y2, both untanglings and the CNAB2 update, inverse
// In the z kernel the two planes of one line are the DCT-III inputs k and nz - k of two real lines, which it
// combines in registers on their way into the tile.  An x tile has the columns ky and ny - ky: the groups k1
// and RA - k1 (0 and RA/2 in the first).
// Six moves of a stage array in place of ten, and two launches in place of four.  Steps before and after:
// 256 x 256 x 384 FP32 185 -> 167 us (78 + 88; the moves alone take 88 at the copy rate), 128 x 96 x 192 FP64
// 61 -> 35, 64^3 FP64 30 -> 13, FP32 24 -> 11.5.  Large boxes are bound by the work between the moves at few
// waves: two blocks a CU in z (58 KB of LDS), one in x (190 registers at 512 threads; held to 128 it spills:
// 256^3 FP32 64 -> 91 us), short ones by the latency of two launches.
// Stage rows (j, x): ny complex values at nsplit_pos; carry [j][kx][t][ky, ny - ky][u] (nsplit_ky).
#pragma once
#include "smx_neumann.h"
#include "smx_split.h"

namespace smx {

template <typename T>
struct SplitNeuArgs {
  cplx<T>*a, *r;                               // stage array and carry, split form, in place
  const cplx<T>*twy, *qtx, *qty, *qtz;         // e^{-2 pi i m/ny}; e^{-i pi k/2n} of the three axes
  PParams<T> p;
};

// Position of (k1, y2): as split_pos, the two k1 of a piece being t and ra - t (0 and ra/2 for t = 0).
__host__ __device__ __forceinline__ int nsplit_pos(int k1, int y2, int ra, int rb) {
  const int g = 2 * k1 >= ra, t = !g ? k1 : (2 * k1 == ra ? 0 : ra - k1);
  return split_pos(2 * t + g, y2, rb);
}
// ky of the first column of pair u of tile t; the second is ny - ky (ny/2 for ky = 0).
__host__ __device__ __forceinline__ int nsplit_ky(int t, int u, int ra, int rb) {
  return t > 0 ? t + ra * u : (2 * u < rb ? ra * u : ra / 2 + ra * (u - rb / 2));
}

// RA of a length (RB = ny / RA); 0: no split.  An x tile has two k1 groups, 2 RB columns, so RB is 8 where
// the z tile can take the rest (sums of the two kernels: 192^3 FP32 50 us with RB 8, 58 with 16; 128 x 96 x
// 192 FP64 31 with 8, 33 with 12, but 96^3 FP64 22 and 20, whose x lines have no plan of E = 8); at 256,
// RA = 32 costs the z kernel what it saves the x kernel.
constexpr int nsplit_ra(int ny, int nx) {
  return ny == 16 || ny == 32 || ny == 48 ? 4
         : ny == 64 || (ny == 96 && nx % 3 == 0) ? 8
         : ny == 96 ? 12
         : ny == 128 || ny == 256 ? 16
         : ny == 192 || ny == 384 ? 24
                                  : 0;
}
// y2 of a z tile: a whole piece where two blocks of it fit a CU, or where two blocks of half a piece do not
// (128^3 FP64 10.3 us, 12.0 with half a piece; 192^3 FP64 41 and 48; 256 x 128 x 256 FP64 with RA 8, 86 KB
// with a whole piece, 46 and 33).
template <typename T>
constexpr int nsplit_ny2(int l, int ra) {
  const int whole = l * (2 * ra + 4) * 2 * (int)sizeof(T), half = l * (ra + 2) * 2 * (int)sizeof(T);
  return whole <= 76 * 1024 || (half > 80 * 1024 && whole + 2 * l * (int)sizeof(T) <= 159 * 1024) ? 4 : 2;
}
// Plan variants: E = 8 where the length has it, except in the z kernel on long lines with two lanes a y line
// (256^3 FP64: 59 us, 62 with E = 8; 128 x 256 x 512 FP32: 46, 59; 256^3 FP32: 49, 39), and in the x kernel
// with 24 columns (128 x 96 x 192 FP64: 20.0, 25.1), with 32 and long lines (256^3 FP64: 140, 146; 128 x 256
// x 512 FP32: 47, 54) and in FP64 at 512 (512 x 128 x 128: 64, 76).
template <typename T, int L>
constexpr int nsplit_zv(int ra) {
  return ra >= 16 && L >= (sizeof(T) == 8 ? 256 : 512) ? 0 : split_v<L>();
}
template <typename T, int L>
constexpr int nsplit_xv(int rb) {
  return rb == 12 || (rb > 8 && L >= (sizeof(T) == 8 ? 256 : 128)) || (sizeof(T) == 8 && L >= 512) ? 0 : split_v<L>();
}

// ---------------------------------------------------------------------------
// z kernel.  Tile: one x, NY2 adjacent y2, every k1 (y1) and plane.  Columns are pairs of real lines of
// neighbouring y1 (of one lane's, P = 2) and equal y2.
template <typename T_, int L_, int RA_, int NY2_ = nsplit_ny2<T_>(L_, RA_), int V_ = nsplit_zv<T_, L_>(RA_),
          int P_ = split_lanes(RA_)>
struct NZ {
  using T = T_;
  static constexpr int L = L_, RA = RA_, NY2 = NY2_, V = V_, P = P_;
  static constexpr int E = PlanV<L, V>::E, TPC = L / E;
  static constexpr int NPR = RA * NY2 / 2, NT = NPR * TPC;
  static constexpr int H = RA / P, HC = H / 2;
  // Tile pitches of the items and of the transform, as in ZS; one in FP32, where the second costs the registers
  // that let a second block of 1024 threads on the CU (256^3: 40 -> 53 us).
  static constexpr int HP = NPR + NY2, FP = sizeof(T) == 8 ? NPR : HP;
  static constexpr int ITEMS = L / 2 * NY2 * P, IPT = (ITEMS + NT - 1) / NT;
  static constexpr int SP = NPR + 1, LDS = L * HP, SLDS = LDS;  // (SP < HP)
  static constexpr int RED = (NT % 64 == 0) ? NT / 64 : NT;
  static constexpr size_t BYTES = (size_t)(LDS + L) * sizeof(cplx<T>) + RED * 8;
  static constexpr bool fits = NT <= 1024 && BYTES <= 160 * 1024;
};

// Byte offset of an item's value k: k1 = k (P = 1), or k + H lo.
template <typename Z>
__device__ __forceinline__ uint32_t nz_leg(int k, int lo, uint32_t step, uint32_t cb) {
  constexpr int RA = Z::RA, H = Z::H;
  if constexpr (Z::P == 2) return k == 0 ? 0u : (uint32_t)(lo ? H - k : k) * step;
  const int g = 2 * k >= RA, t = !g ? k : (2 * k == RA ? 0 : RA - k);
  return (uint32_t)t * step + (uint32_t)(g * kSplitYC) * cb;
}
template <typename Z, typename T>
__device__ __forceinline__ void nz_twiddles(const cplx<T>* __restrict__ qtz, int tid, cplx<T> (*w)[2]) {
#pragma unroll
  for (int it = 0; it < Z::IPT; ++it) {
    const int j = (tid + it * Z::NT) / Z::P / Z::NY2;
    if (tid + it * Z::NT < Z::ITEMS) {
      w[it][0] = qtz[j];
      w[it][1] = qtz[j == 0 ? Z::L / 2 : Z::L - j];
    }
  }
}

// Inverse half: radix RA over k1 of the tile's rows and the DCT-III along z; v receives (psi_a, psi_b) of
// column pair q at z = src(pos_in<inv_last>).  The z twiddles go to twl behind the tile's loads.  w receives
// the thread's items: the lines' cosine coefficients along z at a pair of kz.
template <typename Z, typename TI, typename T = typename Z::T>
__device__ __forceinline__ void nz_inverse_w(const cplx<TI>* src, uint32_t rowb, int rb, cplx<T>* F, cplx<T>* TW,
                                             const cplx<T>* __restrict__ twg, const cplx<T> (*qw)[2], int tid, int q,
                                             int tc, cplx<T>* v, cplx<T> (&w)[Z::IPT][Z::H]) {
  constexpr int L = Z::L;
  constexpr uint32_t CB = sizeof(cplx<TI>);
#pragma unroll
  for (int it = 0; it < Z::IPT; ++it) {  // every load is issued before the first is used
    const int i = tid + it * Z::NT, lo = i % Z::P, c = i / Z::P % Z::NY2, j = i / Z::P / Z::NY2;
    if (i < Z::ITEMS) {
      const uint32_t o = (uint32_t)j * rowb + (uint32_t)(c + lo * kSplitYC) * CB, step = (uint32_t)(2 * rb) * CB;
#pragma unroll
      for (int k = 0; k < Z::H; ++k) {
        const cplx<TI> g = ld_off(src, o + nz_leg<Z>(k, lo, step, CB));
        w[it][k] = mk((T)g.x, (T)g.y);
      }
    }
  }
  const cplx<T>* twl = tw_lds<L, Z::NT>(TW, twg, tid);
#pragma unroll
  for (int it = 0; it < Z::IPT; ++it) {
    const int i = tid + it * Z::NT, lo = i % Z::P, c = i / Z::P % Z::NY2, j = i / Z::P / Z::NY2;
    if (i < Z::ITEMS) {
      if constexpr (Z::P == 2) pair_dft<Z::H, +1, true>(w[it], lo);
      else dft<Z::H, +1>(w[it]);
      cplx<T>* fa = &F[j * Z::HP + lo * Z::HC * Z::NY2 + c];
      cplx<T>* fb = &F[(j == 0 ? L / 2 : L - j) * Z::HP + lo * Z::HC * Z::NY2 + c];
#pragma unroll
      for (int h = 0; h < Z::HC; ++h) {
        const cplx<T> s = mk(w[it][2 * h].x, w[it][2 * h + 1].x);  // the two lines at kz = j ...
        const cplx<T> t = mk(w[it][2 * h].y, w[it][2 * h + 1].y);  // ... and at its partner
        fa[h * Z::NY2] = dct3_in(s, j == 0 ? mk<T>(0, 0) : t, qw[it][0]);
        fb[h * Z::NY2] = dct3_in(t, j == 0 ? t : s, qw[it][1]);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < Z::E; ++e) v[e] = F[Tile<T, L, Z::E, Z::HP>::template pos_in<inv_first<L, Z::V>()>(tc, e) * Z::HP + q];
  InvFFT<T, L, Z::FP, Z::V>::run(v, F, q, tc, twl);
}
template <typename Z, typename TI, typename T = typename Z::T>
__device__ __forceinline__ void nz_inverse(const cplx<TI>* src, uint32_t rowb, int rb, cplx<T>* F, cplx<T>* TW,
                                           const cplx<T>* __restrict__ twg, const cplx<T> (*qw)[2], int tid, int q,
                                           int tc, cplx<T>* v) {
  cplx<T> w[Z::IPT][Z::H];
  nz_inverse_w<Z, TI>(src, rowb, rb, F, TW, twg, qw, tid, q, tc, v, w);
}

// Forward half: the DCT-II along z of the pairs in v and radix RA over y1.
template <typename Z, typename T = typename Z::T>
__device__ __forceinline__ void nz_forward(cplx<T>* v, cplx<T>* dst, uint32_t rowb, int rb, cplx<T>* F,
                                           const cplx<T>* TW, const cplx<T> (*qw)[2], int tid, int q, int tc) {
  constexpr int L = Z::L;
  constexpr uint32_t CB = sizeof(cplx<T>);
  FwdFFT<T, L, Z::FP, Z::V>::run(v, F, q, tc, TW);
  __syncthreads();
  Tile<T, L, Z::E, Z::HP>::template store<fwd_last<L, Z::V>()>(v, F, q, tc);
  __syncthreads();
#pragma unroll
  for (int it = 0; it < Z::IPT; ++it) {
    const int i = tid + it * Z::NT, lo = i % Z::P, c = i / Z::P % Z::NY2, j = i / Z::P / Z::NY2;
    if (i < Z::ITEMS) {
      const cplx<T>* fa = &F[j * Z::HP + lo * Z::HC * Z::NY2 + c];
      const cplx<T>* fb = &F[(j == 0 ? L / 2 : L - j) * Z::HP + lo * Z::HC * Z::NY2 + c];
      cplx<T> w[Z::H];
#pragma unroll
      for (int h = 0; h < Z::HC; ++h) {
        const cplx<T> A = fa[h * Z::NY2], B = fb[h * Z::NY2];
        const cplx<T> s = dct2_out(A, j == 0 ? A : B, qw[it][0]), t = dct2_out(B, j == 0 ? B : A, qw[it][1]);
        w[2 * h] = mk(s.x, t.x);
        w[2 * h + 1] = mk(s.y, t.y);
      }
      if constexpr (Z::P == 2) pair_dft<Z::H, -1, false>(w, lo);
      else dft<Z::H, -1>(w);
      const uint32_t o = (uint32_t)j * rowb + (uint32_t)(c + lo * kSplitYC) * CB, step = (uint32_t)(2 * rb) * CB;
#pragma unroll
      for (int k = 0; k < Z::H; ++k) st_off(dst, o + nz_leg<Z>(k, lo, step, CB), w[k]);
    }
  }
}

template <typename Z>
__global__ __launch_bounds__(Z::NT) void k_nsplit_z(SplitNeuArgs<typename Z::T> s) {
  using T = typename Z::T;
  constexpr int E = Z::E, L = Z::L;
  __shared__ cplx<T> F[Z::LDS];
  __shared__ cplx<T> TW[L];
  __shared__ double red[Z::RED];
  const PParams<T>& p = s.p;
  const int tid = threadIdx.x, q = tid % Z::NPR, tc = tid / Z::NPR;
  const int rb = p.ny / Z::RA;
  int x, yg;
  zs_tile(blockIdx.x, rb / Z::NY2, x, yg);
  const uint32_t rowb = (uint32_t)p.nxy * (uint32_t)sizeof(cplx<T>);
  cplx<T>* base = s.a + (int64_t)x * p.ny + split_pos(0, yg * Z::NY2, rb);
  cplx<T> v[E], qw[Z::IPT][2];
  nz_twiddles<Z>(s.qtz, tid, qw);
  nz_inverse<Z>((const cplx<T>*)base, rowb, rb, F, TW, p.twz, qw, tid, q, tc, v);
  if (p.nl_model == 1) {
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = mk(nonlin3(p, v[e].x), nonlin3(p, v[e].y));
  } else {
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = mk(nonlin5(p, v[e].x), nonlin5(p, v[e].y));
  }
  if (p.partial != nullptr) zs_partial<T, E, Z::NT>(v, red, tid);
  nz_forward<Z>(v, base, rowb, rb, F, TW, qw, tid, q, tc);  // its barriers order red[]
  if (p.partial != nullptr && tid == 0) {
    double t = 0.0;
    for (int w = 0; w < Z::RED; ++w) t += red[w];
    p.partial[blockIdx.x] = t;
  }
}

// Real field (FP64, dense [x][y][z]) of a split-form stage array of type TI: the inverse half alone.
template <typename Z, typename TI>
__global__ __launch_bounds__(Z::NT) void k_nsplit_real(const cplx<TI>* a, double* __restrict__ out, PParams<double> p,
                                                       const cplx<double>* __restrict__ qtz) {
  constexpr int L = Z::L;
  __shared__ cplx<double> F[Z::LDS];
  __shared__ cplx<double> TW[L];
  const int tid = threadIdx.x, q = tid % Z::NPR, tc = tid / Z::NPR;
  const int rb = p.ny / Z::RA;
  int x, yg;
  zs_tile(blockIdx.x, rb / Z::NY2, x, yg);
  cplx<double> v[Z::E], qw[Z::IPT][2];
  nz_twiddles<Z>(qtz, tid, qw);
  nz_inverse<Z>(a + (int64_t)x * p.ny + split_pos(0, yg * Z::NY2, rb), (uint32_t)p.nxy * (uint32_t)sizeof(cplx<TI>), rb,
                F, TW, p.twz, qw, tid, q, tc, v);
  __syncthreads();
#pragma unroll
  for (int e = 0; e < Z::E; ++e)
    F[mk_src(Tile<double, L, Z::E, Z::HP>::template pos_in<inv_last<L, Z::V>()>(tc, e), L) * Z::HP + q] = v[e];
  __syncthreads();
  for (int i = tid; i < Z::NPR * L; i += Z::NT) {  // lanes run along z of one column pair: two coalesced rows
    const int qq = i / L, n = i - qq * L;
    const int c = qq % Z::NY2, h = qq / Z::NY2 % Z::HC, lo = qq / Z::NY2 / Z::HC;
    const int ya = 2 * h * Z::P + lo, yb = ya + Z::P;  // y1 of the two lines
    const cplx<double> w = F[n * Z::HP + qq];
    out[((int64_t)x * p.ny + mk_src(ya * rb + yg * Z::NY2 + c, p.ny)) * L + n] = w.x;
    out[((int64_t)x * p.ny + mk_src(yb * rb + yg * Z::NY2 + c, p.ny)) * L + n] = w.y;
  }
}

// ---------------------------------------------------------------------------
// x kernel.  Tile: one pair of planes, the columns of two k1 groups (of four, RB = 4), every x.
template <typename T_, int L_, int RB_, int V_ = nsplit_xv<T_, L_>(RB_)>
struct NX {
  using T = T_;
  static constexpr int L = L_, RB = RB_, V = V_;
  static constexpr int G = RB == 4 ? 2 : 1, NC = 2 * RB * G, HC = NC / 2;
  static constexpr int E = PlanV<L, V>::E, TPC = L / E, NT = NC * TPC, NCP = NC + 1, NK = NC / RB;
  using AD = RowAddr<NCP>;
  static constexpr int NIT = (L / 2 + 2 * TPC - 1) / (2 * TPC);  // row pairs per thread
  static constexpr size_t BYTES = (size_t)L * (NCP + 2) * sizeof(cplx<T>) + L * sizeof(T);
  static constexpr bool fits = NT <= 1024 && BYTES <= 160 * 1024;
};

template <typename X>
__global__ __launch_bounds__(X::NT) void k_nsplit_x(SplitNeuArgs<typename X::T> s) {
  using T = typename X::T;
  constexpr int L = X::L, RB = X::RB, NC = X::NC, V = X::V, HC = X::HC;
  constexpr int E = X::E, TPC = X::TPC, NT = X::NT, NCP = X::NCP, NIT = X::NIT;
  constexpr uint32_t CB = sizeof(cplx<T>);
  using AD = typename X::AD;
  using TL = Tile<T, L, E, NCP>;
  __shared__ cplx<T> S[L * NCP];
  __shared__ cplx<T> TW[L];
  __shared__ cplx<T> QX[L];
  __shared__ T KX[L];
  const PParams<T>& p = s.p;
  const int tid = threadIdx.x, col = tid % NC, tc = tid / NC;
  const int ra = p.ny / RB, g = p.ny / NC, np = p.nz / 2;
  // tiles of one plane on consecutive slots of one XCD (whole groups of 8 planes; the rest in order)
  int j, bx;
  {
    const int b = blockIdx.x, whole = np / 8 * 8 * g;
    const int i = b >> 3;
    j = b < whole ? i / g * 8 + (b & 7) : b / g;
    bx = b < whole ? i % g : b % g;
  }
  const int ct = bx * X::G + col / (2 * RB), cg = col / RB % 2, y2 = col % RB;
  const int k1 = ct > 0 ? (cg ? ra - ct : ct) : (cg ? ra / 2 : 0);
  const int64_t plane = (int64_t)j * p.nxy;
  const uint32_t rowb = (uint32_t)p.ny * CB;
  const uint32_t aofs = (uint32_t)split_pos(2 * ct + cg, y2, RB) * CB;
  cplx<T>* src = s.a + plane;
  cplx<T>* rb = s.r + plane;
  cplx<T> v[E];
#pragma unroll
  for (int e = 0; e < E; ++e)
    v[e] = ld_off<cplx<T>>(src, (uint32_t)mk_src(TL::template pos_in<fwd_first<L, V>()>(tc, e), L) * rowb + aofs);
  const cplx<T>* twl = tw_lds<L, NT>(TW, p.twx, tid);
  tw_lds<L, NT>(QX, s.qtx, tid);
  for (int i = tid; i < L; i += NT) KX[i] = p.kx[i];
  const cplx<T> tw = s.twy[k1 * y2];  // w_ny^{y2 k1}
  // the thread's pair of columns: ky and ny - ky (0 and ny/2, each its own partner) of planes kz and nz - kz
  const int u = tid % HC % RB, hb = tid % HC / RB, t = bx * X::G + hb, r0 = tid / HC;
  const int kya = nsplit_ky(t, u, ra, RB);
  const bool selfc = kya == 0;
  const int kyb = selfc ? p.ny / 2 : p.ny - kya;
  const bool low = 2 * u < RB;
  const int ca = hb * 2 * RB + (t > 0 || low ? u : RB / 2 + u);
  const int cb = hb * 2 * RB + (t > 0 ? 2 * RB - 1 - u : (low ? (u == 0 ? RB / 2 : RB - u) : 2 * RB - 1 - (u - RB / 2)));
  const cplx<T> wa = s.qty[kya], wb = s.qty[kyb];
  const T kyv[2] = {p.ky[kya], p.ky[kyb]};
  const T kzv[2] = {p.kz[j], p.kz[j == 0 ? np : p.nz - j]};
  const uint32_t rofs = (uint32_t)(t * 2 * RB + u) * CB;
  double nsum = 0.0;
  const bool owner0 = (p.partial != nullptr) && j == 0 && bx == 0;
  if (owner0) nsum = xs_partial_sum<X>(p, S, tid);
#pragma unroll
  for (int e = 0; e < E; ++e) v[e] = cmul(v[e], tw);
  RowFFT<true, T, L, E, AD, -1, typename PlanV<L, V>::Fwd>::run(v, S, col, tc, twl, [&]() { XRow<X, -1>::run(S, tid); });
  // the carry, behind the transform's last reads: a thread's values of it are free, and no store is ahead
  cplx<T> rin[NIT][2][2];
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int i = r0 + it * 2 * TPC;
    if (i < L / 2) {
      const int rows[2] = {i, i == 0 ? L / 2 : L - i};
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          rin[it][a][b] = ld_off<cplx<T>>(rb, (uint32_t)rows[a] * rowb + rofs + (uint32_t)(b * RB) * CB);
    }
  }
  lds_barrier();
#pragma unroll
  for (int e = 0; e < E; ++e) S[AD::at(TL::template pos_in<fwd_last<L, V>()>(tc, e), col)] = v[e];
  lds_barrier();
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int i = r0 + it * 2 * TPC;
    if (i < L / 2) {
      const bool selfr = i == 0;
      const int rows[2] = {i, selfr ? L / 2 : L - i};
      const cplx<T> qa = QX[rows[0]], qb = QX[rows[1]];
      cplx<T> x[2][2];  // [row][column]: REDFT10 along x, then along y
      {
        const cplx<T> a0 = S[AD::at(rows[0], ca)], a1 = S[AD::at(rows[1], ca)];
        const cplx<T> b0 = S[AD::at(rows[0], cb)], b1 = S[AD::at(rows[1], cb)];
        x[0][0] = dct2_out(a0, selfr ? a0 : a1, qa);
        x[1][0] = dct2_out(a1, selfr ? a1 : a0, qb);
        x[0][1] = dct2_out(b0, selfr ? b0 : b1, qa);
        x[1][1] = dct2_out(b1, selfr ? b1 : b0, qb);
      }
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const cplx<T> y0 = x[a][0], y1 = x[a][1];
        x[a][0] = dct2_out(y0, selfc ? y0 : y1, wa);
        x[a][1] = dct2_out(y1, selfc ? y1 : y0, wb);
        const T kxv = KX[rows[a]];
#pragma unroll
        for (int b = 0; b < 2; ++b) {  // cosNoAdvMorph.cpp:431-435, :524-525 with R = C1 psi - dt/2 N_past
          const T kk = kxv * kxv + kyv[b] * kyv[b];
          const T da = kk + kzv[0] * kzv[0] - p.q02, db = kk + kzv[1] * kzv[1] - p.q02;
          const T La = p.eps - p.alpha * da * da, Lb = p.eps - p.alpha * db * db;
          const cplx<T> nn = p.scale * x[a][b], r = rin[it][a][b];
          cplx<T> ps = mk((r.x + (T)3 * p.dtd2 * nn.x) * recip((T)1 - p.dtd2 * La),
                          (r.y + (T)3 * p.dtd2 * nn.y) * recip((T)1 - p.dtd2 * Lb));
          cplx<T> rn = mk(((T)1 + p.dtd2 * La) * ps.x - p.dtd2 * nn.x, ((T)1 + p.dtd2 * Lb) * ps.y - p.dtd2 * nn.y);
          if (a == 0 && b == 0 && owner0 && selfr && selfc) {  // the mean, FP64 (mixed path)
            const double ps0 = (p.mean_state[0] + 3.0 * p.m_dtd2 * (p.m_scale * nsum)) / p.m_c2;
            p.mean_state[0] = p.m_c1 * ps0 - p.m_dtd2 * (p.m_scale * nsum);
            p.mean_state[1] = ps0;
            ps.x = (T)ps0;
            rn.x = (T)p.mean_state[0];
          }
          st_off(rb, (uint32_t)rows[a] * rowb + rofs + (uint32_t)(b * RB) * CB, rn);
          x[a][b] = ps;
        }
        const cplx<T> p0 = x[a][0], p1 = x[a][1];  // REDFT01 inputs along y; the partner of ky = 0 is zero
        x[a][0] = dct3_in(p0, selfc ? mk<T>(0, 0) : p1, wa);
        x[a][1] = dct3_in(p1, selfc ? p1 : p0, wb);
      }
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int c = b == 0 ? ca : cb;
        S[AD::at(rows[0], c)] = dct3_in(x[0][b], selfr ? mk<T>(0, 0) : x[1][b], qa);
        S[AD::at(rows[1], c)] = dct3_in(x[1][b], selfr ? x[1][b] : x[0][b], qb);
      }
    }
  }
  lds_barrier();
#pragma unroll
  for (int e = 0; e < E; ++e) v[e] = S[AD::at(TL::template pos_in<inv_first<L, V>()>(tc, e), col)];
  RowFFT<true, T, L, E, AD, +1, typename PlanV<L, V>::Inv>::run(v, S, col, tc, twl, [&]() { XRow<X, +1>::run(S, tid); });
#pragma unroll
  for (int e = 0; e < E; ++e)
    st_off(src, (uint32_t)mk_src(TL::template pos_in<inv_last<L, V>()>(tc, e), L) * rowb + aofs, cmul(v[e], conjg(tw)));
}

// ---------------------------------------------------------------------------
// Between the two forms, out of place, in FP64.  Rows (j, x) of the split form, two planes of the standard one.
// Rows r0 .. of the split form and their two planes' rows of the standard one, PL, by the first nr threads.
__device__ __forceinline__ void nform_planes(int64_t (*PL)[2], int r0, int nr, int nx, int nz, int ny, int tid) {
  if (tid < nr) {
    const int j = (r0 + tid) / nx, x = r0 + tid - j * nx;
    PL[tid][0] = ((int64_t)j * nx + x) * ny;
    PL[tid][1] = ((int64_t)(j == 0 ? nz / 2 : nz - j) * nx + x) * ny;
  }
}

// To standard as k_form_std, but with the lines' untangling from LDS (ky and ny - ky of a row are two threads')
// and real rows stored 8 bytes a lane (256 x 256 x 384 from FP32: 151 -> 67 us).
template <typename TI, typename TO, int RA, int RB>
__global__ __launch_bounds__(128) void k_nform_std(const TI* __restrict__ in, TO* __restrict__ out, int nx, int nz,
                                                   const cplx<double>* __restrict__ twy,
                                                   const cplx<double>* __restrict__ qty) {
  using C = cplx<double>;
  constexpr int NT = 128, NY = RA * RB, ROWS = NT / RA, N = ROWS * NY, YC = kSplitYC;
  __shared__ C S[N + N / 16];
  __shared__ C TW[NY];
  __shared__ int64_t PL[ROWS][2];  // where the two planes' rows are
  auto at = [](int i) { return i + (i >> 4); };
  const int tid = threadIdx.x, row = tid / RA, k1 = tid - row * RA;
  const int nrows = nx * (nz / 2), r0 = blockIdx.x * ROWS, nr = nrows - r0 < ROWS ? nrows - r0 : ROWS;
  const bool item = row < nr;
  C w[RB];
  if (item) {
    const cplx<TI>* src = reinterpret_cast<const cplx<TI>*>(in) + (int64_t)(r0 + row) * NY + nsplit_pos(k1, 0, RA, RB);
#pragma unroll
    for (int c = 0; c < RB; c += 2) {
      const cplx2<TI> g = *reinterpret_cast<const cplx2<TI>*>(src + c / YC * 2 * YC + c % YC);
      w[c] = mk((double)g.a.x, (double)g.a.y);
      w[c + 1] = mk((double)g.b.x, (double)g.b.y);
    }
  }
  tw_lds<NY, NT>(TW, twy, tid);
  nform_planes(PL, r0, nr, nx, nz, NY, tid);
  __syncthreads();
  if (item) {
#pragma unroll
    for (int c = 1; c < RB; ++c) w[c] = cmul(w[c], TW[k1 * c]);
    dft<RB, -1>(w);
#pragma unroll
    for (int c = 0; c < RB; ++c) S[at(row * NY + k1 + RA * c)] = (0.5 / RB) * w[c];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < (N + NT - 1) / NT; ++u) {
    const int i = tid + u * NT, rr = i / NY, c = i - rr * NY;
    if (rr < nr) {
      const C y = dct2_out(S[at(i)], S[at(rr * NY + (c == 0 ? 0 : NY - c))], qty[c]);
      out[PL[rr][0] + c] = (TO)y.x;
      out[PL[rr][1] + c] = (TO)y.y;
    }
  }
}

// From standard, once after a state is set or loaded: the mirror image, with both sides of memory along the rows and
// every index by constants (256 x 256 x 384 FP32 128 us with divisions at run time, now 78; the carry 80 and 46;
// 256^3 FP64 87 and 54).
template <typename T, int RA, int RB>
__global__ __launch_bounds__(128) void k_nform_split(const T* __restrict__ in, T* __restrict__ out, int nx, int nz,
                                                     const cplx<double>* __restrict__ twy,
                                                     const cplx<double>* __restrict__ qty) {
  using C = cplx<double>;
  constexpr int NT = 128, NY = RA * RB, ROWS = NT / RA, N = ROWS * NY, U = (N + NT - 1) / NT;
  __shared__ C S[N + N / 16];
  __shared__ C TW[NY];
  __shared__ int64_t PL[ROWS][2];
  auto at = [](int i) { return i + (i >> 4); };
  const int tid = threadIdx.x, row = tid / RA, k1 = tid - row * RA;
  const int nrows = nx * (nz / 2), r0 = blockIdx.x * ROWS, nr = nrows - r0 < ROWS ? nrows - r0 : ROWS;
  const bool item = row < nr;
  nform_planes(PL, r0, nr, nx, nz, NY, tid);
  __syncthreads();
  cplx<T> g[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {  // every load is issued before the first is used
    const int i = tid + u * NT, rr = i / NY, c = i - rr * NY;
    if (rr < nr) g[u] = mk(in[PL[rr][0] + c], in[PL[rr][1] + c]);
  }
  tw_lds<NY, NT>(TW, twy, tid);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int i = tid + u * NT;
    if (i < nr * NY) S[at(i)] = mk((double)g[u].x, (double)g[u].y);
  }
  __syncthreads();
  C w[RB];
  if (item) {
#pragma unroll
    for (int c = 0; c < RB; ++c) {
      const int k = k1 + RA * c;
      w[c] = dct3_in(S[at(row * NY + k)], k == 0 ? mk<double>(0, 0) : S[at(row * NY + NY - k)], qty[k]);
    }
    dft<RB, +1>(w);
#pragma unroll
    for (int c = 1; c < RB; ++c) w[c] = cmul(w[c], conjg(TW[k1 * c]));
  }
  __syncthreads();
  if (item) {
#pragma unroll
    for (int c = 0; c < RB; ++c) S[at(row * NY + nsplit_pos(k1, c, RA, RB))] = w[c];
  }
  __syncthreads();
  cplx<T>* dst = reinterpret_cast<cplx<T>*>(out) + (int64_t)r0 * NY;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int i = tid + u * NT;
    if (i < nr * NY) dst[i] = mk((T)S[at(i)].x, (T)S[at(i)].y);
  }
}

// The carry's orders: the pair of planes at ky of the standard form, at (t, ky or ny - ky, u) of the other.
template <typename T, int RA, int RB, bool TO_STD>
__global__ __launch_bounds__(128) void k_nform_perm(const T* __restrict__ in, T* __restrict__ out, int nx, int nz) {
  constexpr int NT = 128, NY = RA * RB, ROWS = NT / RA, N = ROWS * NY, U = (N + NT - 1) / NT;
  __shared__ cplx<T> S[N + N / 16];
  __shared__ int64_t PL[ROWS][2];
  auto at = [](int i) { return i + (i >> 4); };
  auto ky = [](int c) {
    const int k = nsplit_ky(c / (2 * RB), c % RB, RA, RB);
    return c / RB % 2 == 0 ? k : (k == 0 ? NY / 2 : NY - k);
  };
  const int tid = threadIdx.x;
  const int nrows = nx * (nz / 2), r0 = blockIdx.x * ROWS, nr = nrows - r0 < ROWS ? nrows - r0 : ROWS;
  nform_planes(PL, r0, nr, nx, nz, NY, tid);
  __syncthreads();
  const cplx<T>* src = reinterpret_cast<const cplx<T>*>(in) + (int64_t)r0 * NY;
  cplx<T>* dst = reinterpret_cast<cplx<T>*>(out) + (int64_t)r0 * NY;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int i = tid + u * NT, rr = i / NY, c = i - rr * NY;
    if (rr < nr) {
      if constexpr (TO_STD) S[at(rr * NY + ky(c))] = src[i];
      else S[at(i)] = mk(in[PL[rr][0] + c], in[PL[rr][1] + c]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int i = tid + u * NT, rr = i / NY, c = i - rr * NY;
    if (rr < nr) {
      if constexpr (TO_STD) {
        out[PL[rr][0] + c] = S[at(i)].x;
        out[PL[rr][1] + c] = S[at(i)].y;
      } else {
        dst[i] = S[at(rr * NY + ky(c))];
      }
    }
  }
}

}  // namespace smx
