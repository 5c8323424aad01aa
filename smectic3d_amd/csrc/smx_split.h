// smx_split.h -- the periodic step in two launches: the y transform divided between the z and
// the x kernel.
//
// A length-ny transform with ny = RA * RB, y = y1 RB + y2, ky = k1 + RA k2, is
//   X[k1 + RA k2] = sum_y2 w_RB^{y2 k2} w_ny^{y2 k1} ( sum_y1 w_RA^{y1 k1} x[y1 RB + y2] )
// (Cooley and Tukey 1965): radix RA over y1 at fixed y2, then radix RB over y2 at fixed k1.  The z
// kernel holds all y1 of a few y2 (and all z), the x kernel all y2 of a few k1 (and all x), so each
// does its part of the y transform on a tile it has in LDS anyway, and the two y passes, with 4 of
// the step's 10 moves of a stage array through HBM, are gone:
//   k_zsplit  (x, k1 y2, kz) -> (x, k1 y2, kz)   radix RA over k1, z C2R, N(psi), z R2C, radix RA over y1
//   k_xsplit  (x, k1 y2, kz) -> (x, k1 y2, kz)   forward x with radix RB over y2, CNAB2 update, inverse
// Between the two a stage row (kz, x) holds the y2-space, k1-space values in the order of split_pos,
// and the carry R(kx, ky = k1 + RA k2, kz) is at [kz][kx][k1 RB + k2] (the split form; the four-pass
// kernels of smx_periodic.h and the diagnostics use the standard one, ky at its index).
//
// In the z kernel a lane has both lines of a column pair, so that it combines their half spectra into the
// transform's input (and the other way back) in registers; a tile of half spectra, combined as it is read,
// took two reads per value each way (64 -> 59 us at 256^3 FP64, 39.4 -> 37.0 at 192 x 96 x 384).
//
// Measured at 256^3: four passes 213 us FP64 and 112 us FP32 a step; the two kernels 59 + 98 us and
// 33 + 46 us (6 moves of a stage array at the copy rate would take 118 and 59 us).  Smaller boxes gain
// from two launches in place of four as well: 64^3 FP32 3.75 -> 2.56 ms for 200 steps and their checks.
#pragma once
#include "smx_periodic.h"

namespace smx {

// RA of a length (RB = ny / RA); 0: no split.  Both tiles hold NZ RA (2 or 4) / 2 and NX RB values, so
// the two factors are near each other and RB <= 16 (an x tile of 256 x 16 FP64 values is 64 KB).
constexpr int split_ra(int ny) {
  return ny == 16 || ny == 48 ? 4
         : ny == 32 || ny == 64 || ny == 96 || ny == 128 ? 8
         : ny == 192 ? 12
         : ny == 256 ? 16
         : ny == 384 ? 24
                     : 0;
}

// Position of (k1, y2) in a split-form stage row: pieces of YC adjacent y2 of two adjacent k1.  The z
// kernel's tile has every k1 and YC y2, the x kernel's few k1 and every y2, so with either index alone
// fastest one of the two would touch a quarter of each 128-byte line; in this order both use half of
// the lines that they touch.
constexpr int kSplitYC = 4;
__host__ __device__ __forceinline__ int split_pos(int k1, int y2, int rb) {
  constexpr int YC = kSplitYC;
  return (k1 >> 1) * 2 * rb + (y2 / YC) * 2 * YC + (k1 & 1) * YC + y2 % YC;
}
// y2 of a z tile: a whole piece or half of one (the tile's two parities of k1 share a line).  Whole pieces
// on long lines of a power of two (256^3 FP32: 32.9 us, 34.3 with halves; 128^3 FP32 9.7 and 11.4, FP64 15.0
// and 15.2), where two blocks of the tile still fit a CU, and on the shortest, where half a piece would
// leave a wave mostly empty.  Half pieces, twice the blocks, in all others (192^3 FP32 20.4 us, 23.3 with
// whole; 96^3 FP64 10.1 and 11.0; 192 x 96 x 384 FP64 37.0 and 46.8; 64 x 64 x 256 FP64 10.4 and 11.6).
template <typename T>
constexpr int split_ny2(int l, int ra) {
  const bool fp32 = sizeof(T) == 4;
  return (l <= 32 || ra == 4 || (l > 96 && l % 3 != 0 && (fp32 || l <= 128))) && (ra <= 8 || fp32) &&
                 l * (2 * ra + 4) * 2 * (int)sizeof(T) <= 80 * 1024
             ? 4
             : 2;
}
// FP32 halves are 16 bytes: whole pieces also of a large tile, 12 or 24 values of a y line and a long z line, where
// they leave blocks for most of the chip (us with halves and whole: 256 x 192 x 384 66 and 57, 256 x 384 x 192 55 and
// 51, the advected kernels of 256 x 192 x 512 359 + 480 and 321 + 322; but 16 x 192 x 512, 64 whole blocks, a step 29.4 and
// 31.8), not with 16 values (256 x 256 x 384 80 and 93).
template <typename T>
constexpr bool split_whole(int l, int ra) {
  return sizeof(T) == 4 && ((ra == 12 && l >= 384) || (ra == 24 && l >= 192 && l <= 256));
}
constexpr int kSplitWholeBlocks = 192;
// Padding of a z tile's rows of npr values for the items, whose lanes write runs of ny2 columns of successive
// rows: ny2 columns, which lets those runs fall in other banks, or less where a CU has three blocks or fewer and the
// room makes another one fit.
// Rows of 8 more than a multiple of 16 then have one column (none, if that alone leaves one block), rows of 4 more
// none, and fall apart as well.  FP64 z kernels: 256 x 192 x 256 78 us with two blocks a CU, 58 with three; 384 x 384 x
// 128 130 and 86; 384 x 96 x 512 113 with one, 79 with two; FP32 256 x 192 x 256 43 and 32.
template <typename T>
constexpr int split_pad(int l, int npr, int ny2) {
  const auto per_cu = [&](int pad) { return 160 * 1024 / (l * (npr + pad + 1) * 2 * (int)sizeof(T) + 128); };
  const int full = per_cu(ny2);
  if (npr % 16 == 0 || full > 3) return ny2;
  if (npr % 16 == 8) return per_cu(1) > full ? 1 : (full < 2 && per_cu(0) >= 2 ? 0 : ny2);
  return per_cu(0) > full ? 0 : ny2;
}
// Lanes that share one y line in the z kernel (pair_dft): two from radix 16 on, where one lane's 16
// values make its loads the longest part (256^3 FP32: 40.6 -> 34.0 us; 192^3 FP32: 22.3 with one, 27.7).
constexpr int split_lanes(int ra) { return ra >= 16 ? 2 : 1; }

// Plan variants: E = 8 where the length has it; E = 16 for the FP32 z kernel at 256 and 512.
template <int L>
constexpr int split_v() {
  return HasPlanV<L, 1>::value && L >= 64 ? 1 : 0;
}
template <typename T, int L>
constexpr int split_zv() {
  return sizeof(T) == 4 && L >= 256 ? 0 : split_v<L>();
}
// Whether the x kernel reads the carry together with the stage rows.  In short boxes, which are bound by
// latency (64^3 FP32 5.4 -> 4.8 us, 96^3 11.6 -> 10.2); in others the registers cost a block per CU
// (256^3 FP64 102 -> 116 us).
template <typename T, int L>
constexpr bool split_pre() {
  return L <= 96 || (sizeof(T) == 4 && L <= 128);
}
// Columns per x tile: whole k1 groups of RB, rows of 128 bytes or more (96^3 FP32 with 12 columns 10.2
// us, with 24 9.3; FP64 and long lines, whose blocks would pass 512 threads, keep 12).
template <typename T, int L>
constexpr int split_nc(int rb) {
  return rb <= 8 ? 16 : (rb == 12 && sizeof(T) == 4 && L <= 192 ? 24 : rb);
}

template <typename T>
struct SplitArgs {
  cplx<T>* a;               // stage array, split form, in place
  cplx<T>* r;               // carry, split form
  const cplx<T>* twy;       // e^{-2 pi i m/ny}
  PParams<T> p;
};

// ---------------------------------------------------------------------------
// z kernel.  Tile: one x, NY2 adjacent y2, every k1 (y1) and kz.
template <typename T_, int L_, int RA_, int NY2_ = split_ny2<T_>(L_, RA_), int V_ = split_zv<T_, L_>(),
          int P_ = split_lanes(RA_)>
struct ZS {
  using T = T_;
  static constexpr int L = L_, RA = RA_, NY2 = NY2_, V = V_, P = P_;
  static constexpr int E = PlanV<L, V>::E, TPC = L / E;
  static constexpr int NPR = RA * NY2 / 2, NT = NPR * TPC, NZH = L / 2 + 1;
  static constexpr int H = RA / P, HC = H / 2;
  // Tile pitch of the transform, of the items, and of a tile whose columns are read along z (lanes on successive
  // rows, an odd pitch or the items').  Column q: the lines y1 = 2 (q / NY2) and the next, y2 = q % NY2.
  static constexpr int FP = NPR, HP = NPR + split_pad<T>(L, NPR, NY2), SP = NPR + 1;
  // Items of the y part, H values each: one kz, one y2 and (P = 2) one parity of k1, half of the y1.
  static constexpr int ITEMS = NZH * NY2 * P, IPT = (ITEMS + NT - 1) / NT;
  static constexpr int LDS = L * HP, SLDS = L * (HP > SP ? HP : SP);
  static constexpr int RED = (NT % 64 == 0) ? NT / 64 : NT;
  static constexpr bool fits = NT <= 1024 && (size_t)(LDS + L) * sizeof(cplx<T>) + RED * 8 <= 160 * 1024;
};

// Sum of x + y of the E values of every thread, FP64, into red[] (one entry per wave, or per thread
// where the last wave is not full); zs_partial_store adds them after a later barrier.
template <typename T, int E, int NT>
__device__ __forceinline__ void zs_partial(const cplx<T>* v, double* red, int tid) {
  double t[E];
#pragma unroll
  for (int e = 0; e < E; ++e) t[e] = (double)v[e].x + (double)v[e].y;
#pragma unroll
  for (int w = 1; w < E; w *= 2)
#pragma unroll
    for (int e = 0; e + w < E; e += 2 * w) t[e] += t[e + w];
  if constexpr (NT % 64 == 0) {
    const double ws = wave_sum(t[0]);
    if ((tid & 63) == 0) red[tid >> 6] = ws;
  } else {
    red[tid] = t[0];
  }
}

// R(k) <- (R(k) + conj R(-k))/2 on the self-conjugate planes kz = 0 and nz/2 of a split-form carry
// (why: see xpass_tile).  The blocks of one launch share the pairs; each pair is one thread's.
template <typename T>
__device__ __forceinline__ void split_project(cplx<T>* r, const PParams<T>& p, int ra, int blk, int nblk, int tid,
                                              int nt) {
  const int rb = p.ny / ra, nxy = (int)p.nxy;
  for (int i = blk * nt + tid; i < 2 * nxy; i += nblk * nt) {
    const int pl = i >= nxy, j = i - pl * nxy;
    const int kx = j / p.ny, c = j - kx * p.ny, k1 = c / rb, k2 = c - k1 * rb;
    const int mx = kx == 0 ? 0 : p.nx - kx;
    const int m1 = k1 == 0 ? 0 : ra - k1;
    const int m2 = k1 == 0 ? (k2 == 0 ? 0 : rb - k2) : rb - 1 - k2;
    const int m = mx * p.ny + m1 * rb + m2;
    if (m < j) continue;
    cplx<T>* q = r + (pl ? (int64_t)(p.nz / 2) * p.nxy : 0);
    const cplx<T> a = q[j], b = q[m];
    const cplx<T> h = mk((T)0.5 * (a.x + b.x), (T)0.5 * (a.y - b.y));
    q[j] = h;
    q[m] = conjg(h);
  }
}

// The value of the neighbouring lane (lane ^ 1).
__device__ __forceinline__ float lane_xor1(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, true));
}
__device__ __forceinline__ double lane_xor1(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)b, 0xB1, 0xf, 0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), 0xB1, 0xf, 0xf, true);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
// w[y] times e^{SIGN 2 pi i y / R}
template <int R, int SIGN, int Y, int N, typename T>
__device__ __forceinline__ void rot_all(cplx<T>* w) {
  if constexpr (Y < N) {
    w[Y] = rot<R, Y, SIGN>(w[Y]);
    rot_all<R, SIGN, Y + 1, N>(w);
  }
}
// Radix 2 H of one line held by two adjacent lanes: even and odd inputs in, the two halves of the outputs
// out, or (HALVES) the other way round.  Here even and odd k1, and halves of the y1, so SIGN decides.  The
// pair and its neighbours load and store whole lines' halves together, and every thread of the block has
// a part of the work.
template <int H, int SIGN, bool HALVES = (SIGN < 0), typename T>
__device__ __forceinline__ void pair_dft(cplx<T>* w, int lo) {
  const T sgn = lo ? (T)-1 : (T)1;
  auto cross = [&]() {
#pragma unroll
    for (int y = 0; y < H; ++y) {
      const cplx<T> o = mk(lane_xor1(w[y].x), lane_xor1(w[y].y));
      w[y] = mk(o.x + sgn * w[y].x, o.y + sgn * w[y].y);
    }
  };
  if constexpr (!HALVES) {
    dft<H, SIGN>(w);
    if (lo) rot_all<2 * H, SIGN, 0, H>(w);
    cross();
  } else {
    cross();
    if (lo) rot_all<2 * H, SIGN, 0, H>(w);
    dft<H, SIGN>(w);
  }
}

// Byte offset of an item's value k: every other k1 (P = 2) or every k1; step: two k1 apart.
template <typename Z>
__device__ __forceinline__ uint32_t zs_leg(int k, uint32_t step, uint32_t cb) {
  return Z::P == 2 ? (uint32_t)k * step : (uint32_t)(k / 2) * step + (uint32_t)((k & 1) * kSplitYC) * cb;
}

// Inverse half: radix RA over k1 of the tile's rows and the C2R along z; v receives (psi_a, psi_b) of
// the column pair q at z = pos_in<inv_last>.  TI: type of the stage array (float: widened).  kzm: k_z
// table of the spectral d/dz (rows times i k_z, Nyquist +pi/dz, pf3d.cpp:184), or nullptr.  twg: the
// z twiddles in memory, copied to twl behind the tile's loads, or nullptr if they are there.  w receives the
// thread's items: the lines' half spectra along z.
template <typename Z, typename TI, typename T = typename Z::T>
__device__ __forceinline__ void zs_inverse_w(const cplx<TI>* src, uint32_t rowb, int rb, cplx<T>* F,
                                             const cplx<T>* twl, int tid, int q, int tc, cplx<T>* v,
                                             cplx<T> (&w)[Z::IPT][Z::H], const T* kzm, const cplx<T>* twg) {
  constexpr int L = Z::L;
  constexpr uint32_t CB = sizeof(cplx<TI>);
#pragma unroll
  for (int it = 0; it < Z::IPT; ++it) {  // every load is issued before the first is used
    const int i = tid + it * Z::NT, lo = i % Z::P, c = i / Z::P % Z::NY2, m = i / Z::P / Z::NY2;
    if (i < Z::ITEMS) {
      const uint32_t o = (uint32_t)m * rowb + (uint32_t)(c + lo * kSplitYC) * CB, step = (uint32_t)(2 * rb) * CB;
#pragma unroll
      for (int k = 0; k < Z::H; ++k) {
        const cplx<TI> g = ld_off(src, o + zs_leg<Z>(k, step, CB));
        w[it][k] = mk((T)g.x, (T)g.y);
      }
    }
  }
  if (twg != nullptr) tw_lds<L, Z::NT>(const_cast<cplx<T>*>(twl), twg, tid);
#pragma unroll
  for (int it = 0; it < Z::IPT; ++it) {
    const int i = tid + it * Z::NT, lo = i % Z::P, c = i / Z::P % Z::NY2, m = i / Z::P / Z::NY2;
    if (i < Z::ITEMS) {
      if constexpr (Z::P == 2) pair_dft<Z::H, +1>(w[it], lo);
      else dft<Z::H, +1>(w[it]);
      if (kzm != nullptr) {
        const T kz = kzm[m];
#pragma unroll
        for (int k = 0; k < Z::H; ++k) w[it][k] = mk(-kz * w[it][k].y, kz * w[it][k].x);
      }
      // A + iB of two lines at m, and at L - m from the conjugates; only the real parts of kz = 0 and
      // nz/2 enter (the half-complex stage of an FFTW c2r)
      const T im = (m == 0 || m == L / 2) ? (T)0 : (T)1;
      cplx<T>* fa = &F[m * Z::HP + lo * Z::HC * Z::NY2 + c];
      cplx<T>* fb = &F[(m == 0 ? 0 : L - m) * Z::HP + lo * Z::HC * Z::NY2 + c];
#pragma unroll
      for (int h = 0; h < Z::HC; ++h) {
        const cplx<T> A = mk(w[it][2 * h].x, im * w[it][2 * h].y), B = mk(w[it][2 * h + 1].x, im * w[it][2 * h + 1].y);
        fa[h * Z::NY2] = mk(A.x - B.y, A.y + B.x);
        fb[h * Z::NY2] = mk(A.x + B.y, B.x - A.y);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < Z::E; ++e)
    v[e] = F[Tile<T, L, Z::E, Z::HP>::template pos_in<inv_first<L, Z::V>()>(tc, e) * Z::HP + q];
  InvFFT<T, L, Z::FP, Z::V>::run(v, F, q, tc, twl);
}
template <typename Z, typename TI, typename T = typename Z::T>
__device__ __forceinline__ void zs_inverse(const cplx<TI>* src, uint32_t rowb, int rb, cplx<T>* F,
                                           const cplx<T>* twl, int tid, int q, int tc, cplx<T>* v,
                                           const T* kzm = nullptr, const cplx<T>* twg = nullptr) {
  cplx<T> w[Z::IPT][Z::H];
  zs_inverse_w<Z, TI>(src, rowb, rb, F, twl, tid, q, tc, v, w, kzm, twg);
}

// Forward half: the R2C along z of the pairs in v and radix RA over y1 of the half spectra.
template <typename Z, typename T = typename Z::T>
__device__ __forceinline__ void zs_forward(cplx<T>* v, cplx<T>* dst, uint32_t rowb, int rb, cplx<T>* F,
                                           const cplx<T>* twl, int tid, int q, int tc) {
  constexpr int L = Z::L;
  constexpr uint32_t CB = sizeof(cplx<T>);
  FwdFFT<T, L, Z::FP, Z::V>::run(v, F, q, tc, twl);
  __syncthreads();
  Tile<T, L, Z::E, Z::HP>::template store<fwd_last<L, Z::V>()>(v, F, q, tc);
  __syncthreads();
#pragma unroll
  for (int it = 0; it < Z::IPT; ++it) {
    const int i = tid + it * Z::NT, lo = i % Z::P, c = i / Z::P % Z::NY2, m = i / Z::P / Z::NY2;
    if (i < Z::ITEMS) {
      const cplx<T>* fa = &F[m * Z::HP + lo * Z::HC * Z::NY2 + c];
      const cplx<T>* fb = &F[(m == 0 ? 0 : L - m) * Z::HP + lo * Z::HC * Z::NY2 + c];
      cplx<T> w[Z::H];
#pragma unroll
      for (int h = 0; h < Z::HC; ++h) {
        const cplx<T> W = fa[h * Z::NY2], Wm = fb[h * Z::NY2];
        // W = X + iY:  X = (W_k + conj W_{-k})/2,  Y = (W_k - conj W_{-k})/(2i)
        w[2 * h] = mk((T)0.5 * (W.x + Wm.x), (T)0.5 * (W.y - Wm.y));
        w[2 * h + 1] = mk((T)0.5 * (W.y + Wm.y), (T)0.5 * (Wm.x - W.x));
      }
      if constexpr (Z::P == 2) pair_dft<Z::H, -1>(w, lo);
      else dft<Z::H, -1>(w);
      const uint32_t o = (uint32_t)m * rowb + (uint32_t)(c + lo * kSplitYC) * CB, step = (uint32_t)(2 * rb) * CB;
#pragma unroll
      for (int k = 0; k < Z::H; ++k) st_off(dst, o + zs_leg<Z>(k, step, CB), w[k]);
    }
  }
}

// Tile of block bz: x and the first y2.  Blocks of one x on consecutive slots of one XCD (workgroups
// go round the 8 XCDs): they share the 128-byte lines of its rows, whose pieces then meet in one L2.
__device__ __forceinline__ void zs_tile(int bz, int g, int& x, int& yg) {
  const int xcd = bz & 7, i = bz >> 3;
  const int xi = i / g;
  x = xi * 8 + xcd;
  yg = i - xi * g;
}

// nproj leading blocks project R (split_project): the x kernel before left it unprojected, and the
// one behind needs it.
template <typename Z, typename T = typename Z::T>
__device__ __forceinline__ void zsplit_tile(cplx<T>* a, cplx<T>* r, int op, const PParams<T> p, int bx, int nproj) {
  constexpr int E = Z::E, L = Z::L, RA = Z::RA;
  __shared__ cplx<T> F[Z::LDS];
  __shared__ cplx<T> TW[L];
  __shared__ double red[Z::RED];
  const int tid = threadIdx.x, q = tid % Z::NPR, tc = tid / Z::NPR;
  if (bx < nproj) {
    split_project(r, p, RA, bx, nproj, tid, Z::NT);
    return;
  }
  const int bz = bx - nproj;
  const int rb = p.ny / RA;
  int x, yg;
  zs_tile(bz, rb / Z::NY2, x, yg);
  const uint32_t rowb = (uint32_t)p.nxy * (uint32_t)sizeof(cplx<T>);
  cplx<T>* base = a + (int64_t)x * p.ny + split_pos(0, yg * Z::NY2, rb);
  cplx<T> v[E];
  zs_inverse<Z>((const cplx<T>*)base, rowb, rb, F, TW, tid, q, tc, v, (const T*)nullptr, p.twz);
  constexpr int RP = fwd_first<L, Z::V>();
  static_assert(fwd_first<L, Z::V>() == inv_last<L, Z::V>(), "plan symmetry");
  const bool pen = (op == Z_OP_NL) && p.mid > 0 && p.mid < L - 1;
  if (pen) {
    __syncthreads();
    Tile<T, L, E, Z::FP>::template store<RP>(v, F, q, tc);
    __syncthreads();
  }
  if (op == Z_OP_NL && !pen) {
    if (p.nl_model == 1) {
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = mk(nonlin3(p, v[e].x), nonlin3(p, v[e].y));
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = mk(nonlin5(p, v[e].x), nonlin5(p, v[e].y));
    }
  } else if (op == Z_OP_NL) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int n = Tile<T, L, E, Z::FP>::template pos_in<RP>(tc, e);
      T s = nonlin(p, v[e].x), t = nonlin(p, v[e].y);
      if (n == p.mid) {  // pf3dMorph.cpp:572-581
        const cplx<T> lo = F[(n - 1) * Z::FP + q], hi = F[(n + 1) * Z::FP + q];
        s += p.pen * (lo.x - (T)2 * v[e].x + hi.x);
        t += p.pen * (lo.y - (T)2 * v[e].y + hi.y);
      }
      v[e] = mk(s, t);
    }
  }
  if (p.partial != nullptr) zs_partial<T, E, Z::NT>(v, red, tid);
  zs_forward<Z>(v, base, rowb, rb, F, TW, tid, q, tc);  // its barriers order red[]
  if (p.partial != nullptr && tid == 0) {
    double s = 0.0;
    for (int w = 0; w < Z::RED; ++w) s += red[w];
    p.partial[bz] = s;
  }
}
template <typename Z>
__global__ __launch_bounds__(Z::NT) void k_zsplit(SplitArgs<typename Z::T> s, int op, int nproj) {
  zsplit_tile<Z>(s.a, s.r, op, s.p, blockIdx.x, nproj);
}
template <typename Z>
__global__ __launch_bounds__(Z::NT) void k_zsplit_grp(const SplitArgs<typename Z::T>* __restrict__ g, int op,
                                                      int nproj) {
  const SplitArgs<typename Z::T>& b = g[blockIdx.y];
  zsplit_tile<Z>(b.a, b.r, op, b.p, blockIdx.x, nproj);
}

// Real field (FP64, dense [x][y][z]) of a split-form stage array of type TI: the inverse half alone.
template <typename Z, typename TI>
__global__ __launch_bounds__(Z::NT) void k_zsplit_real(const cplx<TI>* a, double* __restrict__ out, PParams<double> p) {
  constexpr int L = Z::L, RA = Z::RA;
  __shared__ cplx<double> F[Z::SLDS];
  __shared__ cplx<double> TW[L];
  const int tid = threadIdx.x, q = tid % Z::NPR, tc = tid / Z::NPR;
  const int rb = p.ny / RA;
  int x, yg;
  zs_tile(blockIdx.x, rb / Z::NY2, x, yg);
  cplx<double> v[Z::E];
  zs_inverse<Z, TI>(a + (int64_t)x * p.ny + split_pos(0, yg * Z::NY2, rb),
                    (uint32_t)p.nxy * (uint32_t)sizeof(cplx<TI>), rb, F, TW, tid, q, tc, v,
                    (const double*)nullptr, p.twz);
  __syncthreads();
  Tile<double, L, Z::E, Z::SP>::template store<inv_last<L, Z::V>()>(v, F, q, tc);
  __syncthreads();
  // lanes run along z of one column pair: two coalesced rows
  for (int i = tid; i < Z::NPR * L; i += Z::NT) {
    const int qq = i / L, n = i - qq * L;
    const int y = 2 * (qq / Z::NY2) * rb + yg * Z::NY2 + qq % Z::NY2;
    const cplx<double> w = F[n * Z::SP + qq];
    double* row = out + ((int64_t)x * p.ny + y) * L;
    row[n] = w.x;
    row[(int64_t)rb * L + n] = w.y;
  }
}

// ---------------------------------------------------------------------------
// x kernel.  Tile: one kz, NC = whole k1 groups of RB columns, every x.
// The transform's first exchange passes through the rows: between its store and its load each thread
// takes the RB columns of one group of a row from the tile, does its part of the y transform and puts
// them back (rowop), which costs one read and one write of the tile and a barrier.
template <bool LB, typename T, int L, int E, typename AD, int SIGN, typename Rad> struct RowFFT;
template <bool LB, typename T, int L, int E, typename AD, int SIGN, int R, int... Rest>
struct RowFFT<LB, T, L, E, AD, SIGN, Radices<R, Rest...>> {
  template <typename F>
  __device__ static __forceinline__ void run(cplx<T>* v, cplx<T>* lds, int col, int tc, const cplx<T>* __restrict__ tw,
                                             F&& rowop) {
    constexpr int TPC = L / E;
#pragma unroll
    for (int u = 0; u < E / R; ++u) dft<R, SIGN>(&v[u * R]);
    tile_barrier<LB>();
#pragma unroll
    for (int u = 0; u < E / R; ++u)
#pragma unroll
      for (int r = 0; r < R; ++r) lds[AD::at((tc + TPC * u) * R + r, col)] = v[u * R + r];
    tile_barrier<LB>();
    rowop();
    tile_barrier<LB>();
    if constexpr (sizeof...(Rest) > 0) {
      TileA<T, L, E, AD>::template load<First<Rest...>::value>(v, lds, col, tc);
      fft_passes<LB, T, L, E, AD, SIGN, R, Rest...>(v, lds, col, tc, tw);
    } else {
      TileA<T, L, E, AD>::template load<R>(v, lds, col, tc);
    }
  }
};

template <typename T_, int L_, int RB_, int NC_ = split_nc<T_, L_>(RB_), int V_ = split_v<L_>(),
          bool PRE_ = split_pre<T_, L_>()>
struct XS {
  using T = T_;
  static constexpr int L = L_, RB = RB_, NC = NC_, V = V_;
  static constexpr bool PRE = PRE_;  // the carry is read with the stage rows
  static constexpr int E = PlanV<L, V>::E, TPC = L / E, NT = NC * TPC, NCP = NC + 1, NK = NC / RB;
  using AD = RowAddr<NCP>;
  static constexpr bool fits =
      NT <= 1024 && (size_t)L * (NCP + 1) * sizeof(cplx<T>) + L * sizeof(T) <= 160 * 1024;
};

// The x tile's part of the y transform on its rows, radix RB between y2 and k2 (SIGN -1: y2 -> k2).
// Lanes run down the rows.  The twiddles w_ny^{y2 k1} are one factor per column, so a thread applies
// its column's in registers as it loads (and, conjugated, as it stores) the stage rows: taken here they
// were 15 LDS reads per row each way (256^3 FP32 47.5 -> 45.9 us, 64^3 4.8 -> 4.4).
template <typename X, int SIGN>
struct XRow {
  using T = typename X::T;
  using AD = typename X::AD;
  static constexpr int L = X::L, RB = X::RB, NK = X::NK, NT = X::NT;
  __device__ static __forceinline__ void run(cplx<T>* S, int tid) {
    for (int i = tid; i < L * NK; i += NT) {
      const int g = i / L, row = i - g * L;
      cplx<T> w[RB];
      cplx<T>* s = &S[AD::at(row, g * RB)];
#pragma unroll
      for (int c = 0; c < RB; ++c) w[c] = s[c];
      dft<RB, SIGN>(w);
#pragma unroll
      for (int c = 0; c < RB; ++c) s[c] = w[c];
    }
  }
};

// Sum of the z kernel's FP64 partials over the block, in a fixed order; S is free.
template <typename X, typename T = typename X::T>
__device__ __forceinline__ double xs_partial_sum(const PParams<T>& p, cplx<T>* S, int tid) {
  double* red = reinterpret_cast<double*>(S);  // NT doubles fit: NT <= L NC
  double s = 0.0;
  for (int i = tid; i < p.npartial; i += X::NT) s += p.partial[i];
  red[tid] = s;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if (tid < w && tid + w < X::NT) red[tid] += red[tid + w];
    __syncthreads();
  }
  return red[0];
}

template <typename X, typename T = typename X::T>
__device__ __forceinline__ void xsplit_tile(cplx<T>* a, cplx<T>* __restrict__ rbuf, const cplx<T>* __restrict__ twy,
                                            const PParams<T> p, int bx, int kz) {
  constexpr int L = X::L, RB = X::RB, NC = X::NC, V = X::V;
  constexpr int E = X::E, TPC = X::TPC, NT = X::NT, NCP = X::NCP, NK = X::NK;
  constexpr uint32_t CB = sizeof(cplx<T>);
  using AD = typename X::AD;
  __shared__ cplx<T> S[L * NCP];
  __shared__ cplx<T> TW[L];
  __shared__ T KX[L];
  const int tid = threadIdx.x, col = tid % NC, tc = tid / NC;
  const int ra = p.ny / RB;
  const int ky = bx * NK + col / RB + ra * (col % RB);
  const int64_t plane = (int64_t)kz * p.nxy;
  const uint32_t rowb = (uint32_t)p.ny * CB;
  const uint32_t cofs = (uint32_t)(bx * NC + col) * CB;  // in the carry's rows
  const uint32_t aofs = (uint32_t)split_pos(bx * NK + col / RB, col % RB, RB) * CB;
  cplx<T>* src = a + plane;
  cplx<T>* rb = rbuf + plane;
  cplx<T> v[E];
#pragma unroll
  for (int e = 0; e < E; ++e)
    v[e] = ld_off<cplx<T>>(src, (uint32_t)Tile<T, L, E, NCP>::template pos_in<fwd_first<L, V>()>(tc, e) * rowb + aofs);
  cplx<T> cr[X::PRE ? E : 1];
  if constexpr (X::PRE) {
#pragma unroll
    for (int e = 0; e < E; ++e)
      cr[e] = ld_off<cplx<T>>(rb, (uint32_t)Tile<T, L, E, NCP>::template pos_in<fwd_last<L, V>()>(tc, e) * rowb + cofs);
  }
  // the tables behind the tile's loads, so that their latencies overlap
  const cplx<T>* twl = tw_lds<L, NT>(TW, p.twx, tid);
  for (int i = tid; i < L; i += NT) KX[i] = p.kx[i];
  const cplx<T> tw = twy[(bx * NK + col / RB) * (col % RB)];  // w_ny^{y2 k1}
  const T kyv = p.ky[ky], kzv = p.kz[kz];
  // FP64 mean mode (mixed path): the block owning k = 0 sums the z kernel's partials.
  double nsum = 0.0;
  const bool owner0 = (p.partial != nullptr) && kz == 0 && bx == 0;
  if (owner0) nsum = xs_partial_sum<X>(p, S, tid);
#pragma unroll
  for (int e = 0; e < E; ++e) v[e] = cmul(v[e], tw);
  RowFFT<true, T, L, E, AD, -1, typename PlanV<L, V>::Fwd>::run(v, S, col, tc, twl, [&]() { XRow<X, -1>::run(S, tid); });
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int kxi = Tile<T, L, E, NCP>::template pos_in<fwd_last<L, V>()>(tc, e);
    const uint32_t o = (uint32_t)kxi * rowb + cofs;
    const T kxv = KX[kxi];
    const T k2 = kxv * kxv + kyv * kyv + kzv * kzv;
    const T d = k2 - p.q02;
    const T aLin = p.eps - p.alpha * d * d;                        // pf3d.cpp:205-206
    const T C1 = (T)1 + p.dtd2 * aLin, C2 = (T)1 - p.dtd2 * aLin;  // :214-215
    const cplx<T> nn = p.scale * v[e];
    // psi_new = (R + 3 dt/2 N)/C2, R' = C1 psi_new - dt/2 N (pf3d.cpp:476-478, as xpass_tile)
    const cplx<T> r = X::PRE ? cr[X::PRE ? e : 0] : ld_off<cplx<T>>(rb, o);
    const T ic2 = recip(C2);
    cplx<T> ps = mk(ic2 * (r.x + (T)3 * p.dtd2 * nn.x), ic2 * (r.y + (T)3 * p.dtd2 * nn.y));
    cplx<T> rn = mk(C1 * ps.x - p.dtd2 * nn.x, C1 * ps.y - p.dtd2 * nn.y);
    if (owner0 && tid == 0 && kxi == 0) {  // k = 0 in FP64
      const double dd = p.m_dtd2, n0 = p.m_scale * nsum;
      const double ps0 = (p.mean_state[0] + 3.0 * dd * n0) / p.m_c2;
      p.mean_state[0] = p.m_c1 * ps0 - dd * n0;
      p.mean_state[1] = ps0;
      ps = mk((T)ps0, (T)0);
      rn = mk((T)p.mean_state[0], (T)0);
    }
    st_off(rb, o, rn);
    v[e] = ps;
  }
  RowFFT<true, T, L, E, AD, +1, typename PlanV<L, V>::Inv>::run(v, S, col, tc, twl, [&]() { XRow<X, +1>::run(S, tid); });
#pragma unroll
  for (int e = 0; e < E; ++e)
    st_off(src, (uint32_t)Tile<T, L, E, NCP>::template pos_in<inv_last<L, V>()>(tc, e) * rowb + aofs,
           cmul(v[e], conjg(tw)));
}
// Tile of linear block b of g column groups a plane: with one k1 per tile, the two tiles that share
// the stage rows' lines are neighbours on one XCD (whole groups of 16 blocks; the rest in order).
template <typename X>
__device__ __forceinline__ void xs_tile(int b, int g, int nzh, int& bx, int& kz) {
  if (X::NK == 1 && b < g * nzh / 16 * 16) b = (b >> 4) * 16 + (b & 7) * 2 + ((b >> 3) & 1);
  kz = b / g;
  bx = b - kz * g;
}
template <typename X>
__global__ __launch_bounds__(X::NT) void k_xsplit(SplitArgs<typename X::T> s) {
  int bx, kz;
  xs_tile<X>(blockIdx.x, s.p.ny / X::NC, s.p.nzh, bx, kz);
  xsplit_tile<X>(s.a, s.r, s.twy, s.p, bx, kz);
}
template <typename X>
__global__ __launch_bounds__(X::NT) void k_xsplit_grp(const SplitArgs<typename X::T>* __restrict__ g) {
  const SplitArgs<typename X::T>& b = g[blockIdx.y];
  int bx, kz;
  xs_tile<X>(blockIdx.x, b.p.ny / X::NC, b.p.nzh, bx, kz);
  xsplit_tile<X>(b.a, b.r, b.twy, b.p, bx, kz);
}

// ---------------------------------------------------------------------------
// Between the two forms.  Rows of ny entries, one per (kz, x).
//   to standard: ky = k1 + RA k2 from radix RB over y2 with the twiddles, divided by RB (the split
//   form's y2-space values are an unnormalised inverse); from standard: the inverse of it.
//   perm: the carry's rows, an order of entries only.
// kmul: k_y table of a standard-form input's d/dy, or nullptr.
enum FormDir { FORM_TO_STD = 0, FORM_FROM_STD = 1, FORM_PERM_TO_STD = 2, FORM_PERM_FROM_STD = 3 };
// To standard, which every diagnostic on the spectrum begins with.  A thread has the RB values of one k1 of a
// row, loads them in pieces of YC and stores them 16 bytes a lane with the lanes along k1: every load of the
// block is in flight at once and nothing goes through LDS but the twiddles, so that the copy runs at the rate
// of its bytes (256^3: FP64 78 -> 52 us, 5.2 TB/s, from FP32 78 -> 40).  In place allowed (TI = T): whole rows per
// block, stored behind a barrier.
// TI: the input's type (float rows widened into an FP64 copy).
template <typename T, int RA, int RB, typename TI = T>
__global__ __launch_bounds__(256) void k_form_std(const cplx<TI>* in, cplx<T>* out, int64_t nrows,
                                                  const cplx<T>* __restrict__ twy) {
  constexpr int NY = RA * RB, ROWS = 256 / RA, YC = kSplitYC;
  __shared__ cplx<T> TW[NY];
  const int tid = threadIdx.x, row = tid / RA, k1 = tid - row * RA;
  const int64_t r = (int64_t)blockIdx.x * ROWS + row;
  const bool item = row < ROWS && r < nrows;
  cplx<T> w[RB];
  if (item) {
    const cplx<TI>* src = in + r * NY + split_pos(k1, 0, RB);
#pragma unroll
    for (int c = 0; c < RB; c += 2) {
      const cplx2<TI> g = *reinterpret_cast<const cplx2<TI>*>(src + c / YC * 2 * YC + c % YC);
      w[c] = mk((T)g.a.x, (T)g.a.y);
      w[c + 1] = mk((T)g.b.x, (T)g.b.y);
    }
  }
  tw_lds<NY, 256>(TW, twy, tid);
  __syncthreads();  // the table; and in place, every read of the rows
  if (!item) return;
#pragma unroll
  for (int c = 1; c < RB; ++c) w[c] = cmul(w[c], TW[k1 * c]);
  dft<RB, -1>(w);
  cplx<T>* dst = out + r * NY + k1;
#pragma unroll
  for (int c = 0; c < RB; ++c) dst[RA * c] = (T)(1.0 / RB) * w[c];
}

// From standard, once after a state is set or loaded: the mirror image, loads along k1 and stores in pieces (256^3
// FP64 70 us through LDS on both sides, now 58; FP32 31 and 26).
template <typename T, int RA, int RB>
__global__ __launch_bounds__(256) void k_form_split(const cplx<T>* in, cplx<T>* out, int64_t nrows,
                                                    const cplx<T>* __restrict__ twy, const T* __restrict__ kmul) {
  constexpr int NY = RA * RB, ROWS = 256 / RA, YC = kSplitYC;
  __shared__ cplx<T> TW[NY];
  const int tid = threadIdx.x, row = tid / RA, k1 = tid - row * RA;
  const int64_t r = (int64_t)blockIdx.x * ROWS + row;
  const bool item = row < ROWS && r < nrows;
  cplx<T> w[RB];
  if (item) {
    const cplx<T>* src = in + r * NY + k1;
#pragma unroll
    for (int c = 0; c < RB; ++c) w[c] = src[RA * c];
    if (kmul != nullptr) {  // i k_y of the spectral d/dy (pf3d.cpp:405)
#pragma unroll
      for (int c = 0; c < RB; ++c) {
        const T k = kmul[k1 + RA * c];
        w[c] = mk(-k * w[c].y, k * w[c].x);
      }
    }
  }
  tw_lds<NY, 256>(TW, twy, tid);
  __syncthreads();  // the table; and in place, every read of the rows
  if (!item) return;
  dft<RB, +1>(w);
#pragma unroll
  for (int c = 1; c < RB; ++c) w[c] = cmul(w[c], conjg(TW[k1 * c]));
  cplx<T>* dst = out + r * NY + split_pos(k1, 0, RB);
#pragma unroll
  for (int c = 0; c < RB; c += 2)
    *reinterpret_cast<cplx2<T>*>(dst + c / YC * 2 * YC + c % YC) = cplx2<T>{w[c], w[c + 1]};
}

// The carry's orders.
template <typename T, int RA, int RB, bool TO_STD>
__global__ __launch_bounds__(256) void k_form_perm(const cplx<T>* in, cplx<T>* out, int64_t nrows) {
  constexpr int NY = RA * RB, ROWS = 1024 / NY, N = ROWS * NY;
  __shared__ cplx<T> S[N + N / 16];
  auto at = [](int i) { return i + (i >> 4); };
  const int tid = threadIdx.x;
  const int64_t r0 = (int64_t)blockIdx.x * ROWS;
  const int n = (int)(nrows - r0 < ROWS ? nrows - r0 : ROWS) * NY;
  const cplx<T>* src = in + r0 * NY;
  cplx<T>* dst = out + r0 * NY;
#pragma unroll
  for (int u = 0; u < (N + 255) / 256; ++u)
    if (const int i = tid + u * 256; i < n) S[at(i)] = src[i];
  __syncthreads();
#pragma unroll
  for (int u = 0; u < (N + 255) / 256; ++u)
    if (const int i = tid + u * 256; i < n) {
      const int c = i % NY;
      dst[i] = S[at(i - c + (TO_STD ? c % RA * RB + c / RA : c / RB + RA * (c % RB)))];
    }
}

}  // namespace smx
