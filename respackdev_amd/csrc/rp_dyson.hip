// Dyson step of calc_eps_rpa / calc_eps_rpa_q_0 (chiqw_sub.F:386-568) in FP64
// on gfx950: eps_GG' = delta - 2 chi_GG' 4pi/(|q+G||q+G'|) (head, wings and
// the Drude term at q = 0), then eps^-1 for every frequency of the batch.
//
// The inversion is Gauss-Jordan with partial pivoting by |Re|+|Im| (the pivot
// rule of LAPACK's izamax in zgetrf, which the reference calls through
// invZGE.F90:1-23), blocked by panels: one workgroup per matrix factors a panel (for
// n <= 768 32 columns in registers, else up to 16 in LDS), a batched kernel applies
// the panel's transform to all other columns (for n <= 768 in the same launch as the
// factoring of the next panel), and a final kernel puts the columns in order.
#include <algorithm>
#include <utility>

#include "rp_common.h"
#include "rp_kernels.h"

namespace rp {

// eps[b][j][i] (column-major per matrix), b = dir*nen + w.
__global__ void k_eps_build(const double2* __restrict__ chi, const double* __restrict__ qn, int n,
                            int nen, int q0, int g0, const double* __restrict__ wd,
                            const double2* __restrict__ em, double delt,
                            double2* __restrict__ eps) {
  const int b = blockIdx.y;
  const int j = blockIdx.z;
  const double tpi = 2.0 * 3.141592653589793238462643383279502884;
  const double2* c = chi + ((size_t)b * n + j) * n;
  double2* e = eps + ((size_t)b * n + j) * n;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    double cx = 2.0 * c[i].x, cy = 2.0 * c[i].y;  // spin factor, chiqw_sub.F:413
    double vx, vy;
    if (!q0) {
      vx = cx * 2.0 * tpi / qn[i] / qn[j];
      vy = cy * 2.0 * tpi / qn[i] / qn[j];
      e[i] = i == j ? make_double2(1.0 - vx, -vy) : make_double2(-vx, -vy);
    } else {
      if (i == j && i == g0) {
        const int dir = b / nen, w = b % nen;
        double om = em[w].x;
        if (om == 0.0) om = 1.0e-5;
        const double d2 = wd[dir] * wd[dir];
        // CMPLX(x,y) without KIND: the Drude term is rounded to single precision
        const float drx = (float)(-d2 / (om * om + delt * delt));
        const float dry = (float)(delt * d2 / (om * om * om + om * delt * delt));
        e[i] = make_double2(1.0 - cx * 2.0 * tpi + (double)drx, -cy * 2.0 * tpi + (double)dry);
      } else if (i == j) {
        vx = cx * 2.0 * tpi / qn[i] / qn[j];
        vy = cy * 2.0 * tpi / qn[i] / qn[j];
        e[i] = make_double2(1.0 - vx, -vy);
      } else if (i == g0) {
        e[i] = make_double2(-cx * 2.0 * tpi / qn[j], -cy * 2.0 * tpi / qn[j]);
      } else if (j == g0) {
        e[i] = make_double2(-cx * 2.0 * tpi / qn[i], -cy * 2.0 * tpi / qn[i]);
      } else {
        e[i] = make_double2(-cx * 2.0 * tpi / qn[i] / qn[j], -cy * 2.0 * tpi / qn[i] / qn[j]);
      }
    }
  }
}

__device__ inline double cabs1(double2 z) { return fabs(z.x) + fabs(z.y); }

// acc + a b and acc - a b for complex FP64 as four fused multiply-adds each
// (a product's two terms, each folded into the accumulator).
__device__ __forceinline__ double2 cfma(double2 acc, double2 a, double2 b) {
  return make_double2(fma(a.x, b.x, fma(-a.y, b.y, acc.x)), fma(a.x, b.y, fma(a.y, b.x, acc.y)));
}
__device__ __forceinline__ double2 cfms(double2 acc, double2 a, double2 b) {
  return make_double2(fma(-a.x, b.x, fma(a.y, b.y, acc.x)), fma(-a.x, b.y, fma(-a.y, b.x, acc.y)));
}

// Largest panel width; panel rows moved by the pivoting of one panel: at most
// the nb panel rows plus nb others.
constexpr int kPanelMax = 16;
constexpr int kMoveMax = 2 * kPanelMax;
// Per matrix the panel kernel leaves {count, dst[kMoveMax], src[kMoveMax]}.
constexpr int kMoveInts = 1 + 2 * kMoveMax;

// Blocked Gauss-Jordan.  The nb pivot steps of panel [c0, c0+nb) are
// elementary transforms E_k that differ from the identity only in column k;
// their product differs from the identity only in the panel columns, and
// running the in-place Gauss-Jordan steps on the panel columns alone leaves
// exactly those columns W in the panel.  Every other column j then becomes
//   a'(:,j) = P a(:,j) with the panel rows zeroed + W (P a)(panel rows, j),
// P the panel's row interchanges: one rank-nb update.

// One workgroup per matrix: the panel (n x nb, FP64 complex) is factored in
// LDS; row interchanges are applied to the panel and recorded as a move list
// for the update kernel.  LDS: nb*n double2 + n ints.
__global__ void __launch_bounds__(1024) k_gj_panel(double2* __restrict__ a, int n, int c0, int nb,
                                                   int* __restrict__ ipiv, int* __restrict__ moves,
                                                   int* __restrict__ status) {
  extern __shared__ double2 lds[];
  double2* P = lds;                      // P[l*n + i] = a(i, c0+l)
  int* orig = (int*)(P + (size_t)nb * n);  // orig[i]: original row now in row i
  __shared__ double wv[16];
  __shared__ int wi[16];
  __shared__ double2 prow[kPanelMax];
  __shared__ int nmove;
  __shared__ int singular;
  const int b = blockIdx.x, tid = threadIdx.x, nt = blockDim.x;
  double2* m = a + (size_t)b * n * n;
  for (int l = 0; l < nb; ++l)
    for (int i = tid; i < n; i += nt) P[(size_t)l * n + i] = m[i + (size_t)n * (c0 + l)];
  for (int i = tid; i < n; i += nt) orig[i] = i;
  if (tid == 0) { nmove = 0; singular = 0; }
  __syncthreads();
  for (int l = 0; l < nb; ++l) {
    const int c = c0 + l;
    const double2* col = P + (size_t)l * n;
    // pivot: largest |Re|+|Im| in rows c..n-1, first index on ties (izamax)
    double best = -1.0;
    int bi = n;
    for (int i = c + tid; i < n; i += nt) {
      const double v = cabs1(col[i]);
      if (v > best) { best = v; bi = i; }
    }
    for (int off = 32; off > 0; off >>= 1) {
      const double v2 = __shfl_xor(best, off);
      const int i2 = __shfl_xor(bi, off);
      if (v2 > best || (v2 == best && i2 < bi)) { best = v2; bi = i2; }
    }
    if ((tid & 63) == 0) { wv[tid >> 6] = best; wi[tid >> 6] = bi; }
    __syncthreads();
    if (tid == 0) {
      for (int w = 1; w < nt / 64; ++w)
        if (wv[w] > best || (wv[w] == best && wi[w] < bi)) { best = wv[w]; bi = wi[w]; }
      if (bi >= n) bi = c;  // no candidate compared (NaN column): keep row c, as izamax does
      wi[0] = bi;
      ipiv[(size_t)b * n + c] = bi;
      const int t = orig[c];
      orig[c] = orig[bi];
      orig[bi] = t;
    }
    __syncthreads();
    const int p = wi[0];
    if (p != c && tid < nb) {
      double2* cl = P + (size_t)tid * n;
      const double2 t = cl[c];
      cl[c] = cl[p];
      cl[p] = t;
    }
    __syncthreads();
    const double2 piv = col[c];
    if (piv.x == 0.0 && piv.y == 0.0) {
      if (tid == 0) { atomicOr(status, 4); singular = 1; }
      break;  // uniform: every thread reads the same pivot
    }
    // pivot row c scaled (its column l becomes 1/piv)
    if (tid < nb) {
      const zd pinv = mkz(1.0, 0.0) / mkz(piv.x, piv.y);
      const double2 v = P[(size_t)tid * n + c];
      const zd u = tid == l ? pinv : mkz(v.x, v.y) * pinv;
      prow[tid] = make_double2(u.x, u.y);
    }
    __syncthreads();
    for (int i = tid; i < n; i += nt) {
      if (i == c) {
        for (int q = 0; q < nb; ++q) P[(size_t)q * n + i] = prow[q];
      } else {
        const double2 t = col[i];
        for (int q = 0; q < nb; ++q) {
          double2* e = P + (size_t)q * n + i;
          const double2 v = q == l ? make_double2(0.0, 0.0) : *e;
          *e = cfms(v, t, prow[q]);
        }
      }
    }
    __syncthreads();
  }
  for (int l = 0; l < nb; ++l)
    for (int i = tid; i < n; i += nt) m[i + (size_t)n * (c0 + l)] = P[(size_t)l * n + i];
  // move list: the nb panel rows first (in order), then other rows whose
  // content changed
  int* mv = moves + (size_t)b * kMoveInts;
  if (tid < nb) {
    mv[1 + tid] = c0 + tid;
    mv[1 + kMoveMax + tid] = orig[c0 + tid];
  }
  for (int i = tid; i < n; i += nt) {
    if ((i < c0 || i >= c0 + nb) && orig[i] != i) {
      const int e = nb + atomicAdd(&nmove, 1);
      mv[1 + e] = i;
      mv[1 + kMoveMax + e] = orig[i];
    }
  }
  __syncthreads();
  if (tid == 0) mv[0] = singular ? -1 : nb + nmove;
}

// ---------------------------------------------------------------------------
// n <= 768: steps of 32 columns.  Each launch applies the rank-32 transform of
// one 32-column panel to every other column; one block per matrix brings the
// next panel up to date and factors it in the same launch (look-ahead), as two
// halves of 16 columns in registers: half A, half B after A's transform, then A
// after B's.  The transform of the two halves together differs from the identity
// in the panel's columns only, so every other column j becomes
//   a'(:,j) = P a(:,j) with the panel rows zeroed + W (P a)(panel rows, j),
// W the panel's final columns and P the panel's row interchanges (B's act on
// rows below A's panel rows only, so A's transform commutes past them).  The last
// panel is as narrow as what is left of the columns.
//
// The panel blocks are the critical path: 32 column steps one after the other,
// each about 2400 clocks of latency (pivot search 300, reciprocal 200, offering the
// candidates' rows and meeting at the barrier 800, comparing them 300, the rank-1
// update 700 to 850).  A thread holds R rows (256 R >= n), so that a block has four
// waves, one per SIMD, which meet quickly and take the update's time together.
// Rows are not exchanged between threads: a thread keeps the number lr of the
// matrix row that its values are (-1: no row), and an interchange swaps the
// numbers.  Per launch, 16 to 24 matrices, with a thread per row, two barriers per
// column and the update on the vector unit before: NG 106, first panel 64 -> 49 us,
// a step 59 -> 35; NG 586, 100 -> 85 and 146 -> 120 us.  The last panel in the same
// way instead of by k_gj_panel and k_gj_update: NG 17, all of it, 75 -> 28 us; NG 586
// 107 -> 38 us of one step that has no next panel.
constexpr int kSuper = 32;
constexpr int kHalf = 16;
constexpr int kMoveMax32 = 2 * kSuper;           // panel rows and rows they displaced
constexpr int kMoveInts32 = 1 + 2 * kMoveMax32;  // {count, dst[64], src[64]}
constexpr int kGjThreads = 256;
constexpr int kGjRows = 768;

typedef double d4 __attribute__((ext_vector_type(4)));

struct GjShared {
  // every wave's candidate for the pivot, by the parity of the column: |Re|+|Im|, the
  // row's number, its reciprocal and its other columns
  double2 wv[2][2];
  int4 wi[2];
  double2 rowp[2][4][kHalf];
  int orig[kGjRows];   // the row whose content is now in row i: by the panel, by its half B
  int orig2[kGjRows];
  short slot[kGjRows];  // where row i comes from: -1 itself, -2 zero (panel row), e: vals[e]
  double2 vals[kMoveMax32][kSuper];  // old values of the moved rows
  int dst[kMoveMax32], src[kMoveMax32];
  int nm;
  int singular;
};

// A double moved across lanes by DPP (two 32-bit moves; every lane has a source).
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const int lo = (int)(unsigned)u, hi = (int)(unsigned)(u >> 32);
  const unsigned lo2 = (unsigned)__builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xf, 0xf, false);
  const unsigned hi2 = (unsigned)__builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((unsigned long long)hi2 << 32) | lo2);
}

__device__ __forceinline__ double readlane_d(double v, int l) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), l);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Lane Q of every row of 16 lanes, in all of them.
template <int Q>
__device__ __forceinline__ double2 gj_bcast(double2 v) {
  return make_double2(__builtin_amdgcn_update_dpp(0.0, v.x, 0x150 + Q, 0xf, 0xf, false),
                      __builtin_amdgcn_update_dpp(0.0, v.y, 0x150 + Q, 0xf, 0xf, false));
}

// Columns 1.. of the rows less f times the pivot row (entry q in lane q), moved up
// by one.
template <int R, int... Q>
__device__ __forceinline__ void gj_rank1(std::integer_sequence<int, Q...>,
                                         double2 (&r)[R][kHalf], const double2 (&f)[R], double2 v) {
  (
      [&] {
        const double2 u = gj_bcast<Q + 1>(v);
#pragma unroll
        for (int k = 0; k < R; ++k) r[k][Q] = cfms(r[k][Q + 1], f[k], u);
      }(),
      ...);
}

// 1/z by Smith's scaling without a branch.
__device__ __forceinline__ double2 gj_inv(double2 z) {
  const bool xb = fabs(z.x) >= fabs(z.y);
  const double g = xb ? z.x : z.y, l = xb ? z.y : z.x;
  const double q = l / g, t = 1.0 / fma(l, q, g);
  return xb ? make_double2(t, -q * t) : make_double2(q * t, -t);
}

// The step of column c of a half panel.  The column is in r[.][0], the others
// follow in turn; the step leaves them moved up by one and its own column last, so
// that one loop body of constant register indices serves all columns.  The reciprocal
// of every thread's own candidate is formed while the search runs, which waits on
// latency; only the winner's is used.  Every wave offers its candidate's whole row
// before the one barrier of the step.  A zero pivot sets the status bit and
// sh.singular and the steps go on (on values that are then discarded): every
// thread runs the same steps and meets the same barriers.
template <int R>
__device__ __forceinline__ void gj_step(double2 (&r)[R][kHalf], int (&lr)[R], GjShared& sh, int n,
                                        int c, int* __restrict__ status) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int par = c & 1;
  // pivot: largest |Re|+|Im| in rows c..n-1, first row on ties (izamax); -1: none
  double ob = -1.0;
  int ol = n;
  double2 z = make_double2(1.0, 0.0);
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const double v = fabs(r[k][0].x) + fabs(r[k][0].y);
    const bool g = (lr[k] >= c) & ((v > ob) | ((v == ob) & (lr[k] < ol)));
    ob = g ? v : ob;
    ol = g ? lr[k] : ol;
    z.x = g ? r[k][0].x : z.x;
    z.y = g ? r[k][0].y : z.y;
  }
  const double2 zi = gj_inv(z);
  // wave maximum: butterfly within rows of 16 lanes (DPP), then the four rows
  double best = ob;
  best = fmax(best, dpp_d<0xB1>(best));   // quad_perm [1,0,3,2]
  best = fmax(best, dpp_d<0x4E>(best));   // quad_perm [2,3,0,1]
  best = fmax(best, dpp_d<0x124>(best));  // row_ror:4
  best = fmax(best, dpp_d<0x128>(best));  // row_ror:8
  best = fmax(fmax(readlane_d(best, 0), readlane_d(best, 16)),
              fmax(readlane_d(best, 32), readlane_d(best, 48)));
  const unsigned long long at = __ballot(ob == best);
  int row = __builtin_amdgcn_readlane(ol, __ffsll(at) - 1);
  if (best >= 0.0)
    for (unsigned long long m = at & (at - 1); m; m &= m - 1)  // ties
      row = min(row, __builtin_amdgcn_readlane(ol, __ffsll(m) - 1));
  // one lane of the wave, or none (a row number is in one lane only; n in none)
#pragma unroll
  for (int k = 0; k < R; ++k)
    if (lr[k] == row) {
      double2* o = sh.rowp[par][wave];
      o[0] = zi;
#pragma unroll
      for (int q = 1; q < kHalf; ++q) o[q] = r[k][q];
    }
  if (lane == 0) {
    ((double*)sh.wv[par])[wave] = best;
    ((int*)&sh.wi[par])[wave] = row;
  }
  __syncthreads();
  const double2 w01 = sh.wv[par][0], w23 = sh.wv[par][1];
  const int4 wi = sh.wi[par];
  const bool b1 = (w01.y > w01.x) | ((w01.y == w01.x) & (wi.y < wi.x));
  const bool b3 = (w23.y > w23.x) | ((w23.y == w23.x) & (wi.w < wi.z));
  const double va = b1 ? w01.y : w01.x, vb = b3 ? w23.y : w23.x;
  const int pa = b1 ? wi.y : wi.x, pb = b3 ? wi.w : wi.z;
  const bool bb = (vb > va) | ((vb == va) & (pb < pa));
  best = bb ? vb : va;
  int p = bb ? pb : pa;
  // lane l of a row of 16 lanes reads entry l and the others get it by DPP: read by
  // every lane, an entry costs each wave a read of LDS (first panel of NG 586:
  // 94 us so, 86 this way)
  double2 v = sh.rowp[par][bb ? 2 + b3 : (int)b1][lane & 15];
  if (best < 0.0) {  // no candidate compared (NaN column): keep row c, all becomes NaN
    p = c;
    v.x = v.y = __builtin_nan("");
  }
  if (best == 0.0 && threadIdx.x == 0) {
    atomicOr(status, 4);
    sh.singular = 1;
  }
#pragma unroll
  for (int k = 0; k < R; ++k)
    // the pivot row becomes row c, scaled: zero less the row times -1/pivot
    if (lr[k] == p)
#pragma unroll
      for (int q = 0; q < kHalf; ++q) r[k][q] = make_double2(0.0, 0.0);
  const double2 pinv = gj_bcast<0>(v);
  double2 f[R];  // what multiplies the pivot row
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const double2 g = cfma(make_double2(0.0, 0.0), r[k][0], pinv);
    const bool is = lr[k] == p;
    f[k] = make_double2(is ? -pinv.x : g.x, is ? -pinv.y : g.y);
    lr[k] = is ? c : lr[k] == c ? p : lr[k];  // row c's content is row p's now
  }
  gj_rank1(std::make_integer_sequence<int, kHalf - 1>{}, r, f, v);
#pragma unroll
  for (int k = 0; k < R; ++k) r[k][kHalf - 1] = make_double2(-f[k].x, -f[k].y);
}

// Factors columns [c, c + w), w <= 16, in registers and puts them back; map[i]
// becomes the row whose content is in row i.  Ends with a barrier.
template <int R>
__device__ __forceinline__ void gj_half(GjShared& sh, int* map, double2* m, int n, int c, int w,
                                        int* __restrict__ status) {
  double2 r[R][kHalf];
  int lr[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int i = threadIdx.x + kGjThreads * k;
    lr[k] = i < n ? i : -1;
#pragma unroll
    for (int q = 0; q < kHalf; ++q)
      r[k][q] = i < n && q < w ? m[i + (size_t)n * (c + q)] : make_double2(0.0, 0.0);
  }
#pragma unroll 1
  for (int l = 0; l < w; ++l) gj_step<R>(r, lr, sh, n, c + l, status);
  // column l is now in r[.][16 - w + l]
#pragma unroll
  for (int k = 0; k < R; ++k)
    if (lr[k] >= 0) {
      map[lr[k]] = threadIdx.x + kGjThreads * k;
#pragma unroll
      for (int q = 0; q < kHalf; ++q)
        if (q >= kHalf - w) m[lr[k] + (size_t)n * (c + q - (kHalf - w))] = r[k][q];
    }
  __syncthreads();
}

// The move list of the rows that map moves, the nb panel rows [c0, c0 + nb)
// first, into sh.dst/src/nm.  Ends with a barrier.
__device__ __forceinline__ void gj_list(GjShared& sh, const int* map, int n, int c0, int nb) {
  if (threadIdx.x == 0) sh.nm = nb;
  if ((int)threadIdx.x < nb) {
    sh.dst[threadIdx.x] = c0 + threadIdx.x;
    sh.src[threadIdx.x] = map[c0 + threadIdx.x];
  }
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += kGjThreads)
    if ((i < c0 || i >= c0 + nb) && map[i] != i) {
      const int e = atomicAdd(&sh.nm, 1);  // at most nb of them
      sh.dst[e] = i;
      sh.src[e] = map[i];
    }
  __syncthreads();
}

// Columns [cj, cj + nt) of m, nt <= 16 CT, after the transform of the panel
// [ck, ck + w), w <= 4 KQ, with the move list in sh: C = P a with the panel rows
// zeroed, plus W times the panel rows of P a, on the matrix cores (FP64
// 16x16x4, four real products per complex one).  A wave takes tiles of 16 rows, W and
// C from memory with the next tile's in flight.  On the vector unit every fourth multiply-add needs one of
// the panel rows' values broadcast from LDS.  NG 586, 32 columns of a block: 38 us, of which 17 are the products at the
// rate of the matrix cores.  Begins with writes to LDS that earlier readers must be done with,
// ends with a barrier.
template <int KQ, int CT>
__device__ __forceinline__ void gj_apply(GjShared& sh, double2* m, int n, int ck, int w, int cj,
                                         int nt) {
  constexpr int CW = 16 * CT;
  const int nm = sh.nm;
  for (int x = threadIdx.x; x < nm * CW; x += kGjThreads) {
    const int e = x / CW, t = x % CW;
    sh.vals[e][t] = t < nt ? m[sh.src[e] + (size_t)n * (cj + t)] : make_double2(0.0, 0.0);
  }
  for (int i = threadIdx.x; i < n; i += kGjThreads) sh.slot[i] = -1;
  __syncthreads();
  if ((int)threadIdx.x < nm) sh.slot[sh.dst[threadIdx.x]] = (int)threadIdx.x < w ? -2 : threadIdx.x;
  __syncthreads();
  const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4;
  // loads without conditions, at clamped addresses: what a row or column takes
  // instead of its own value is put in when the value is used
  double2 wn[KQ], cn[CT][4];
  int sn = -1;
  auto load = [&](int tile) {
    const int i = min(16 * tile + lo, n - 1);
    sn = sh.slot[i];
#pragma unroll
    for (int k = 0; k < KQ; ++k) wn[k] = m[i + (size_t)n * (ck + min(4 * k + hi, w - 1))];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        cn[ct][v] = m[i + (size_t)n * (cj + min(16 * ct + hi + 4 * v, nt - 1))];
  };
  const int ntile = (n + 15) / 16;
  int tile = threadIdx.x >> 6;
  if (tile < ntile) load(tile);
  for (; tile < ntile; tile += kGjThreads / 64) {
    double2 wc[KQ];
    d4 re[CT], im[CT];
#pragma unroll
    for (int k = 0; k < KQ; ++k) {
      const bool in = 4 * k + hi < w;
      wc[k] = make_double2(in ? wn[k].x : 0.0, in ? wn[k].y : 0.0);
    }
    const int slot = sn;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        re[ct][v] = slot == -2 ? 0.0 : cn[ct][v].x;
        im[ct][v] = slot == -2 ? 0.0 : cn[ct][v].y;
      }
    if (__ballot(slot >= 0) != 0) {  // few tiles
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const double2 o = sh.vals[max(slot, 0)][16 * ct + hi + 4 * v];
          re[ct][v] = slot >= 0 ? o.x : re[ct][v];
          im[ct][v] = slot >= 0 ? o.y : im[ct][v];
        }
    }
    if (tile + kGjThreads / 64 < ntile) load(tile + kGjThreads / 64);
#pragma unroll
    for (int k = 0; k < KQ; ++k) {
      double2 v[CT];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        v[ct] = 4 * k + hi < w ? sh.vals[4 * k + hi][16 * ct + lo] : make_double2(0.0, 0.0);
        re[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(v[ct].x, wc[k].x, re[ct], 0, 0, 0);
        im[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(v[ct].x, wc[k].y, im[ct], 0, 0, 0);
      }
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        re[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(-v[ct].y, wc[k].y, re[ct], 0, 0, 0);
        im[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(v[ct].y, wc[k].x, im[ct], 0, 0, 0);
      }
    }
    const int i = 16 * tile + lo;
    if (i < n)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int t = 16 * ct + hi + 4 * v;
          if (t < nt) m[i + (size_t)n * (cj + t)] = make_double2(re[ct][v], im[ct][v]);
        }
  }
  __syncthreads();
}

// Factors the panel [c, c + w), w <= 32, of one matrix, its columns up to date
// in m.  Leaves the panel's final columns in m, its move list in mv (count -1 after
// a zero pivot) and in perm[i] the row of the given matrix that is now row i.
template <int R>
__device__ __forceinline__ void gj_panel32(GjShared& sh, double2* m, int n, int c, int w,
                                           int* __restrict__ perm, int* __restrict__ mv,
                                           int* __restrict__ status) {
  const int wa = min(w, kHalf), wb = w - wa;
  if (c == 0)
    for (int i = threadIdx.x; i < n; i += kGjThreads) perm[i] = i;
  if (threadIdx.x == 0) sh.singular = 0;
  gj_half<R>(sh, sh.orig, m, n, c, wa, status);
  if (wb > 0) {
    gj_list(sh, sh.orig, n, c, wa);
    gj_apply<kHalf / 4, 1>(sh, m, n, c, wa, c + wa, wb);
    gj_half<R>(sh, sh.orig2, m, n, c + wa, wb, status);
    gj_list(sh, sh.orig2, n, c + wa, wb);
    gj_apply<kHalf / 4, 1>(sh, m, n, c + wa, wb, c, wa);
  }
  if (sh.singular) {  // uniform: set before the barriers above
    if (threadIdx.x == 0) mv[0] = -1;
    return;
  }
  int o[R], pn[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int i = threadIdx.x + kGjThreads * k;
    if (i < n) {
      o[k] = sh.orig[wb > 0 ? sh.orig2[i] : i];
      pn[k] = perm[o[k]];
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int i = threadIdx.x + kGjThreads * k;
    if (i < n) {
      sh.orig[i] = o[k];
      perm[i] = pn[k];
    }
  }
  __syncthreads();
  gj_list(sh, sh.orig, n, c, w);
  if ((int)threadIdx.x < sh.nm) {
    mv[1 + threadIdx.x] = sh.dst[threadIdx.x];
    mv[1 + kMoveMax32 + threadIdx.x] = sh.src[threadIdx.x];
  }
  if (threadIdx.x == 0) mv[0] = sh.nm;
}

// The first panel: one block per matrix.
template <int R>
__global__ void __launch_bounds__(kGjThreads, R < 3 ? 2 : 1)
    k_gj_first(double2* __restrict__ a, int n, int* __restrict__ perm, int* __restrict__ moves,
               int* __restrict__ status) {
  __shared__ GjShared sh;
  const int b = blockIdx.x;
  gj_panel32<R>(sh, a + (size_t)b * n * n, n, 0, min(n, kSuper), perm + (size_t)b * n,
                moves + (size_t)b * kMoveInts32, status);
}

// One step: the transform of panel k (columns [ck, ck + w), move list moves_k)
// on every other column and, when wn > 0, the factoring of panel k + 1, columns
// [ck + 32, ck + 32 + wn).  Blocks [0, nbatch) (wn > 0) are panel blocks.  Every
// other block updates up to 32 columns of one matrix outside both panels, ngroups
// groups per matrix.  The two kinds touch disjoint columns and read panel k's
// columns only, so nothing in the launch waits for anything else.  With nbatch a
// multiple of 8 the update blocks of matrix b run on XCD b mod 8 (blocks are dealt
// to the XCDs round-robin), so each XCD's L2 holds its matrices' panels.
template <int R>
__global__ void __launch_bounds__(kGjThreads, R < 3 ? 2 : 1)
    k_gj_step32(double2* __restrict__ a, int n, int ck, int w, int wn, int nbatch, int ngroups,
                int* __restrict__ perm, const int* __restrict__ moves_k,
                int* __restrict__ moves_next, int* __restrict__ status) {
  __shared__ GjShared sh;
  const bool panel = wn > 0 && (int)blockIdx.x < nbatch;
  int b, cj, nt;
  if (panel) {
    b = blockIdx.x;
    cj = ck + w;
    nt = wn;
  } else {
    const int u = (int)blockIdx.x - (wn > 0 ? nbatch : 0);
    int t;
    if (nbatch % 8 == 0) {
      const int x = u % 8, s = u / 8;
      b = x + 8 * (s / ngroups);
      t = s % ngroups;
    } else {
      b = u / ngroups;
      t = u % ngroups;
    }
    const int skip = w + wn;      // columns [ck, ck + skip) are not in the groups
    const int t0 = t * kSuper;    // groups never straddle ck (multiples of 32)
    cj = t0 < ck ? t0 : t0 + skip;
    nt = min(kSuper, n - skip - t0);
  }
  double2* m = a + (size_t)b * n * n;
  const int* mv = moves_k + (size_t)b * kMoveInts32;
  const int nm = mv[0];
  if (nm < 0) {  // a zero pivot earlier (the host reports it): nothing more for this matrix
    if (panel && threadIdx.x == 0) moves_next[(size_t)b * kMoveInts32] = -1;
    return;  // uniform: every thread read the same word
  }
  if ((int)threadIdx.x < nm) {
    sh.dst[threadIdx.x] = mv[1 + threadIdx.x];
    sh.src[threadIdx.x] = mv[1 + kMoveMax32 + threadIdx.x];
  }
  if (threadIdx.x == 0) sh.nm = nm;
  __syncthreads();
  gj_apply<kSuper / 4, 2>(sh, m, n, ck, w, cj, nt);
  if (panel)  // uniform per block
    gj_panel32<R>(sh, m, n, cj, nt, perm + (size_t)b * n, moves_next + (size_t)b * kMoveInts32,
                  status);
}

// The columns back in the given matrix's order: with row i of P a the row perm[i]
// of a, column i of (P a)^-1 is column perm[i] of a^-1.  grid (ceil(n / 8),
// nbatch): a block moves eight rows through LDS.
constexpr int kPermRows = 8;
__global__ void __launch_bounds__(512) k_gj_colperm(double2* __restrict__ a, int n,
                                                    const int* __restrict__ perm) {
  extern __shared__ double2 lds[];
  const int b = blockIdx.y, row = blockIdx.x * kPermRows + (threadIdx.x % kPermRows);
  double2* m = a + (size_t)b * n * n;
  for (int x = threadIdx.x; x < n * kPermRows; x += 512)
    if (row < n) lds[x] = m[row + (size_t)n * (x / kPermRows)];
  __syncthreads();
  for (int x = threadIdx.x; x < n * kPermRows; x += 512)
    if (row < n) m[row + (size_t)n * perm[(size_t)b * n + x / kPermRows]] = lds[x];
}

// Rank-nb update of every column outside the panel.  grid: (ceil((n-nb)/TJ),
// nbatch), 256 threads; workgroup = TJ whole columns of one matrix, so the
// reads of moved rows (staged in LDS before the barrier) never race with
// another workgroup's writes.
constexpr int kTJ = 16;
__global__ void __launch_bounds__(256) k_gj_update(double2* __restrict__ a, int n, int c0, int nb,
                                                   const int* __restrict__ moves) {
  __shared__ double2 vals[kMoveMax][kTJ];
  __shared__ int dst[kMoveMax];
  const int b = blockIdx.y, tid = threadIdx.x;
  double2* m = a + (size_t)b * n * n;
  const int* mv = moves + (size_t)b * kMoveInts;
  const int nm = mv[0];
  if (nm < 0) return;  // singular pivot: the host reports it
  const int nrest = n - nb;
  const int jt0 = blockIdx.x * kTJ;
  const int ntj = min(kTJ, nrest - jt0);
  if (tid < nm) dst[tid] = mv[1 + tid];
  for (int e = tid; e < nm * kTJ; e += blockDim.x) {
    const int mi = e / kTJ, t = e % kTJ;
    if (t < ntj) {
      const int jj = jt0 + t, j = jj < c0 ? jj : jj + nb;
      vals[mi][t] = m[mv[1 + kMoveMax + mi] + (size_t)n * j];
    }
  }
  __syncthreads();
  const double2* W = m + (size_t)n * c0;
  for (int i = tid; i < n; i += blockDim.x) {
    double2 w[kPanelMax];
#pragma unroll
    for (int q = 0; q < kPanelMax; ++q)
      if (q < nb) w[q] = W[i + (size_t)n * q];
    const bool inpanel = i >= c0 && i < c0 + nb;
    int slot = -1;
    if (!inpanel)
      for (int e = nb; e < nm; ++e)
        if (dst[e] == i) slot = e;
    for (int t = 0; t < ntj; ++t) {
      const int jj = jt0 + t, j = jj < c0 ? jj : jj + nb;
      double2* out = m + i + (size_t)n * j;
      double2 acc = inpanel ? make_double2(0.0, 0.0) : (slot >= 0 ? vals[slot][t] : *out);
#pragma unroll
      for (int q = 0; q < kPanelMax; ++q)
        if (q < nb) acc = cfma(acc, w[q], vals[q][t]);
      *out = acc;
    }
  }
}

// Undo the row interchanges: swap columns c and ipiv[c] for c = n-1 .. 0.
__global__ void __launch_bounds__(256) k_gj_colswap(double2* __restrict__ a, int n,
                                                    const int* __restrict__ ipiv) {
  const int b = blockIdx.x;
  double2* m = a + (size_t)b * n * n;
  for (int c = n - 1; c >= 0; --c) {
    const int p = ipiv[(size_t)b * n + c];
    if (p != c && p >= 0 && p < n)  // a singular matrix leaves later entries unset
      for (int i = threadIdx.x; i < n; i += blockDim.x) {
        double2 t = m[i + (size_t)n * c];
        m[i + (size_t)n * c] = m[i + (size_t)n * p];
        m[i + (size_t)n * p] = t;
      }
    __syncthreads();
  }
}

// kappa[b] = max_j sum_i |a_b(i, j)| (the 1-norm of each matrix of the batch).
// grid: (ceil(n / 4), nbatch) blocks of 256: one wave per column, its lanes
// reading consecutive rows; the column sums meet in kappa[b] through a 64-bit
// atomic maximum on the bit patterns (non-negative doubles order as their
// bits).  kappa must start at zero.
__global__ void __launch_bounds__(256) k_norm1(const double2* __restrict__ a, int n,
                                               unsigned long long* __restrict__ kappa) {
  const int b = blockIdx.y, j = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (j >= n) return;  // uniform per wave
  const double2* col = a + ((size_t)b * n + j) * n;
  double s = 0.0;
  for (int i = lane; i < n; i += 64) {
    const double2 z = col[i];
    s += sqrt(z.x * z.x + z.y * z.y);
  }
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
  if (lane == 0) atomicMax(kappa + b, __double_as_longlong(s));
}

void launch_norm1(const double2* a, int n, int nbatch, double* kappa, hipStream_t s) {
  launch_zero(kappa, sizeof(double) * (size_t)nbatch, s);
  hipLaunchKernelGGL(k_norm1, dim3((n + 3) / 4, nbatch), dim3(256), 0, s, a, n,
                     (unsigned long long*)kappa);
  RP_HIP(hipGetLastError());
}

void launch_eps_build(const double2* chi, const double* qn, int n, int nbatch, int nen, int q0,
                      int g0, const double* wd, const double2* em, double delt, double2* eps,
                      hipStream_t s) {
  dim3 grid((n + 255) / 256, nbatch, n);
  hipLaunchKernelGGL(k_eps_build, grid, dim3(256), 0, s, chi, qn, n, nen, q0, g0, wd, em, delt, eps);
  RP_HIP(hipGetLastError());
}

// Two move lists per matrix: the fused step reads panel k's while its panel
// blocks write panel k+1's.
size_t gauss_jordan_work_ints(int nbatch) { return 2 * (size_t)nbatch * kMoveInts32; }

template <int R>
static void launch_gj32(double2* a, int n, int nbatch, int* perm, int* work, int* status,
                        hipStream_t s) {
  auto moves = [&](int k) { return work + (size_t)(k & 1) * nbatch * kMoveInts32; };
  hipLaunchKernelGGL(k_gj_first<R>, dim3(nbatch), dim3(kGjThreads), 0, s, a, n, perm, moves(0),
                     status);
  for (int k = 0, ck = 0; ck < n; ++k, ck += kSuper) {
    const int w = std::min(kSuper, n - ck), wn = std::min(kSuper, n - ck - w);
    const int ngroups = (n - w - wn + kSuper - 1) / kSuper;
    const int nblk = (wn > 0 ? nbatch : 0) + nbatch * ngroups;
    if (nblk > 0)
      hipLaunchKernelGGL(k_gj_step32<R>, dim3(nblk), dim3(kGjThreads), 0, s, a, n, ck, w, wn, nbatch,
                         ngroups, perm, (const int*)moves(k), moves(k + 1), status);
  }
}

// ipiv: n ints per matrix; work: gauss_jordan_work_ints(nbatch).
void launch_gauss_jordan(double2* a, int n, int nbatch, int* ipiv, int* work, int* status,
                         hipStream_t s) {
  if (n <= kGjRows) {
    RP_CHECK(n >= 1, "Dyson: empty matrix");
    if (n <= kGjThreads) launch_gj32<1>(a, n, nbatch, ipiv, work, status, s);
    else if (n <= 2 * kGjThreads) launch_gj32<2>(a, n, nbatch, ipiv, work, status, s);
    else launch_gj32<3>(a, n, nbatch, ipiv, work, status, s);
    const size_t lds = sizeof(double2) * kPermRows * n;
    if (lds > 65536)
      RP_HIP(hipFuncSetAttribute((const void*)k_gj_colperm,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k_gj_colperm, dim3((n + kPermRows - 1) / kPermRows, nbatch), dim3(512), lds,
                       s, a, n, (const int*)ipiv);
    RP_HIP(hipGetLastError());
    return;
  }
  // move list of panel number k: work + (k & 1) * nbatch * kMoveInts
  auto moves = [&](int k) { return work + (size_t)(k & 1) * nbatch * kMoveInts; };
  int c0 = 0, panel = 0;
  // panels in LDS, as many columns as fit next to the row map, at most 16, then a
  // rank-nb update
  const size_t budget = 160 * 1024 - 1024 - sizeof(int) * (size_t)n;
  const int nb = (int)std::min<size_t>(kPanelMax, budget / (sizeof(double2) * (size_t)n));
  RP_CHECK(nb >= 1, "Dyson: matrix too large for the LDS panel");
  int maxlds = 0;
  for (; c0 < n; ++panel) {
    const int w = std::min(nb, n - c0);
    const size_t lds = sizeof(double2) * (size_t)w * n + sizeof(int) * (size_t)n;
    if ((int)lds > maxlds && lds > 65536) {
      RP_HIP(hipFuncSetAttribute((const void*)k_gj_panel,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
      maxlds = (int)lds;
    }
    hipLaunchKernelGGL(k_gj_panel, dim3(nbatch), dim3(1024), lds, s, a, n, c0, w, ipiv,
                       moves(panel), status);
    if (n - w > 0)
      hipLaunchKernelGGL(k_gj_update, dim3((n - w + kTJ - 1) / kTJ, nbatch), dim3(256), 0, s, a, n,
                         c0, w, (const int*)moves(panel));
    c0 += w;
  }
  hipLaunchKernelGGL(k_gj_colswap, dim3(nbatch), dim3(256), 0, s, a, n, (const int*)ipiv);
  RP_HIP(hipGetLastError());
}

}  // namespace rp
