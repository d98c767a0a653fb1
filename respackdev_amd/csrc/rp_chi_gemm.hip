// chi_GG'(q,w) = sum_K conj(A[K][G]) d[w][K] A[K][G'] on gfx950 MFMA.
//
// This is the accumulation of chiqw.F:1397-1410 restated as a rank-K update
// per frequency (K = pair*NTK + k), a = A[K][G], b = d A[K][G'],
//   Re chi += Re a Re b + Im a Im b,   Im chi += Re a Im b - Im a Re b.
//
// Workgroup: 256 threads, tile 64 G x 64 G' for one frequency.  Precisions:
//   FP64   k_chi_f64: v_mfma_f64_16x16x4f64, FP64 accumulators, the complex
//          product as three real ones, the tile's 16-blocks dealt to the waves.
//   FP32   k_chi_gemm: v_mfma_f32_16x16x4f32, 2x2 waves of 2x2 blocks; one real
//          product of twice the K, whose k-slots hold (Re a | Im a) against
//          (Re b | Im b) for the real part and (Im b | -Re b) for the imaginary
//          part; FP32 accumulators flushed into FP64 ones every kFlush chunks.
// (The split-BF16 precision has its own kernel, k_chi_bf16x3.)
// The K range may be split over gridDim.z; partial tiles are summed in fixed
// order by k_chi_reduce (deterministic), which also divides by the volume.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "rp_common.h"
#include "rp_kernels.h"

namespace rp {

typedef double d4v __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));

constexpr int kTile = 64;   // G and G' per workgroup
constexpr int kKC = 32;     // complex K rows per LDS chunk
constexpr int kLdsRow = kKC + 2;
constexpr int kFlush = 32;  // chunks per FP32 -> FP64 flush (1024 K)

__device__ inline void stage_chunk(const float2* __restrict__ A, size_t lda, size_t K0, int g0,
                                   int h0, const double2* __restrict__ dw, float2 (*sL)[kLdsRow],
                                   float2 (*sR)[kLdsRow], double2* sD) {
  const int t = threadIdx.x;
#pragma unroll
  for (int e = 0; e < (kTile * kKC) / 256; ++e) {
    int idx = t + 256 * e;
    int kk = idx / kTile, gg = idx % kTile;
    const float2* row = A + (K0 + kk) * lda;
    sL[gg][kk] = row[g0 + gg];
    sR[gg][kk] = row[h0 + gg];
  }
  if (t < kKC) sD[t] = dw[K0 + t];
}

// One output tile in FP32: a K-chunk of 32 complex rows of both panels is
// staged in LDS (transposed to [G][K]) together with the 32 weights, which are
// applied to the right panel as it is read.  out: partial[z][w][ng][ng] with
// element (G, G') at out[... + G' * ng + G] (Fortran chiqw(ig,jg,ie) order).
__global__ void __launch_bounds__(256) k_chi_gemm(const float2* __restrict__ A, size_t lda,
                                                  const double2* __restrict__ dw, size_t ldd,
                                                  size_t kchunks_per_split, size_t kchunks,
                                                  int ng, int ntile, int nen, int cross,
                                                  double2* __restrict__ out) {
  __shared__ float2 sL[kTile][kLdsRow];
  __shared__ float2 sR[kTile][kLdsRow];
  __shared__ double2 sD[kKC];
  const int2 tg = chi_tile_of((int)blockIdx.x, ntile, cross);
  const int tm = tg.x, tn = tg.y;
  const int g0 = tm * kTile, h0 = tn * kTile;
  const int w = blockIdx.y;
  const int z = blockIdx.z;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int li = lane & 15, q = lane >> 4;
  const int part = q >> 1;  // 0: real-part k-slots, 1: imaginary-part k-slots
  const double2* dww = dw + (size_t)w * ldd;
  const size_t c_begin = (size_t)z * kchunks_per_split;
  size_t c_end = c_begin + kchunks_per_split;
  if (c_end > kchunks) c_end = kchunks;

  // block validity (skip 16x16 blocks entirely outside [0, ng))
  bool rowok[2], colok[2];
  for (int b = 0; b < 2; ++b) {
    rowok[b] = g0 + wm * 32 + b * 16 < ng;
    colok[b] = h0 + wn * 32 + b * 16 < ng;
  }

  double accd_re[2][2][4], accd_im[2][2][4];
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b)
      for (int v = 0; v < 4; ++v) accd_re[a][b][v] = accd_im[a][b][v] = 0.0;

  f4v acc_re[2][2], acc_im[2][2];
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b) acc_re[a][b] = acc_im[a][b] = f4v{0, 0, 0, 0};
  const int h = q & 1;
  int since = 0;
  for (size_t c = c_begin; c < c_end; ++c) {
    stage_chunk(A, lda, c * kKC, g0, h0, dww, sL, sR, sD);
    __syncthreads();
#pragma unroll 4
    for (int s = 0; s < 16; ++s) {
      const int kl = h * 16 + s;
      float L[2], Rre[2], Rim[2];
      const float dx = (float)sD[kl].x, dy = (float)sD[kl].y;
      for (int b = 0; b < 2; ++b) {
        float2 la = sL[wm * 32 + b * 16 + li][kl];
        L[b] = part ? la.y : la.x;
        float2 ra = sR[wn * 32 + b * 16 + li][kl];
        float bx = dx * ra.x - dy * ra.y;
        float by = dx * ra.y + dy * ra.x;
        Rre[b] = part ? by : bx;
        Rim[b] = part ? -bx : by;
      }
      for (int a = 0; a < 2; ++a) {
        if (!rowok[a]) continue;
        for (int b = 0; b < 2; ++b) {
          if (!colok[b]) continue;
          acc_re[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(L[a], Rre[b], acc_re[a][b], 0, 0, 0);
          acc_im[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(L[a], Rim[b], acc_im[a][b], 0, 0, 0);
        }
      }
    }
    __syncthreads();
    if (++since == kFlush || c + 1 == c_end) {
      since = 0;
      for (int a = 0; a < 2; ++a)
        for (int b = 0; b < 2; ++b) {
          for (int v = 0; v < 4; ++v) {
            accd_re[a][b][v] += (double)acc_re[a][b][v];
            accd_im[a][b][v] += (double)acc_im[a][b][v];
          }
          acc_re[a][b] = acc_im[a][b] = f4v{0, 0, 0, 0};
        }
    }
  }

  // epilogue: the FP32 MFMA leaves C[4*(lane>>4)+v][lane&15] of a 16x16 block
  // in element v of a lane (checked on gfx950)
  double2* o = out + ((size_t)z * nen + w) * (size_t)ng * ng;
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b)
      for (int v = 0; v < 4; ++v) {
        const int gi = g0 + wm * 32 + a * 16 + 4 * q + v;
        const int hj = h0 + wn * 32 + b * 16 + li;
        if (gi < ng && hj < ng)
          o[(size_t)hj * ng + gi] = make_double2(accd_re[a][b][v], accd_im[a][b][v]);
      }
}

// One output tile in FP64.  With b = d a(G') the complex product conj(a) b is
// three real ones (three real MFMAs per block and 4 K where the direct form
// needs four):
//   T1 = ar bi,  T2 = ai br,  T3 = (ar + ai)(br + bi),
//   Im = T1 - T2,  Re = T3 - T1 - T2.
// T1 and T2 have terms of either sign (the phase of a row of A is its
// eigenvectors' arbitrary one) and stay of the order of Im, so that Im carries no
// rounding of the many times larger Re.  (With T1 = ar br, T2 = ai bi and
// T3 = (ar - ai)(br + bi), T1 - T2 is small and T1, T2 are half of Re each: Im is
// then off by three to five times as much.)
// FP64 MFMAs and FP64 vector instructions share one unit per SIMD (run
// together they reach 58 TFLOP/s, the MFMAs alone 79), so every vector
// operation on the operands costs matrix time: the three left and three right
// planes of a chunk are formed once per workgroup as it is staged (10 vector
// operations per staged element pair against 192 MFMA flops per element of the
// 64-wide tile) and the loop over the chunk is LDS reads and MFMAs only.
// Planes are [k][64 + 16]: the four k of a read fall on both halves of the
// banks.  The loads of the next chunk are in flight during the MFMAs.
//
// Bound by that unit.  NG 441, K 112500, 32 frequencies (5.6 TFLOP): 64.8 ms,
// 67 TFLOP/s executed (the direct form with the weights applied on every read:
// 108.5 ms).  Four workgroups per CU hide the staging, hence 8 K per chunk and
// 128 registers: three (more registers, 8 K) 68.3 ms, two (16 K) 71 ms, two with
// 128 x 64 tiles and fewer vector operations 75.6 ms, two double-buffered 78 ms.
// Error against long double, each part by its own norm, at that size: Re 7e-16 to
// 1e-15, Im 1.3e-15 to 3.1e-15 (direct form 5e-15 to 7e-15 and 1.0e-14; the other
// three products 3.2e-15 to 1.6e-14 for Im); K 1296 to 6144, NG 81 to 126: Re 2.0e-16,
// Im 2.9e-16 to 4.7e-16 (2.0e-16 and 4.1e-16 to 6.2e-16; 1.0e-15 to 1.4e-15).
//
// The right block is the MFMA's first operand, so that D(row, col) =
// (G', G) and the lanes of a result run along G, the fastest index of out.
// The 16-blocks of [0, ng) are dealt evenly to the ntile tiles of an axis (four
// at most: 10 blocks are 3 + 3 + 4, not 4 + 4 + 2), and a tile's blocks to its
// waves so that the busiest has the fewest (4x4: 2x2 each; 3x3: three columns
// of three).  Which wave takes which part rotates with the workgroup so that
// the idler parts spread over the SIMDs.
constexpr int kF64KC = 8;                // K rows per chunk
constexpr int kF64Row = kTile + 16;      // doubles per plane row
constexpr int kF64Plane = kF64KC * kF64Row;

template <int NR, int NC>
__device__ __forceinline__ void f64_chunk(const double* pl, const double* pr, int li, int lk,
                                          d4v (&acc)[3][4]) {
#pragma unroll
  for (int k0 = 0; k0 < kF64KC; k0 += 4)
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      double l[NR], r[NC];
#pragma unroll
      for (int b = 0; b < NC; ++b) r[b] = pr[p * kF64Plane + (k0 + lk) * kF64Row + li + 16 * b];
#pragma unroll
      for (int a = 0; a < NR; ++a) l[a] = pl[p * kF64Plane + (k0 + lk) * kF64Row + li + 16 * a];
#pragma unroll
      for (int a = 0; a < NR; ++a)
#pragma unroll
        for (int b = 0; b < NC; ++b)
          acc[p][a * NC + b] =
              __builtin_amdgcn_mfma_f64_16x16x4f64(r[b], l[a], acc[p][a * NC + b], 0, 0, 0);
    }
}

// HEAD: the row and the column of G = 0 of one direction at q = 0, whose column
// of A is H.  The right columns are then c = (type, frequency), b = d_w H for
// the column (type 0) and conj(d_w) H for the row (type 1, conjugated when
// merged): every frequency in one product of NG x 2 nen x K instead of the
// tiles of that row and column at each frequency.  out: partial[z][c][ng].
template <bool HEAD>
__global__ void __launch_bounds__(256, 4) k_chi_f64(const float2* __restrict__ A, size_t lda,
                                                    const double2* __restrict__ dw, size_t ldd,
                                                    size_t chunks_per_split, size_t nchunks,
                                                    int ng, int ntile, int nen,
                                                    const float2* __restrict__ H,
                                                    double2* __restrict__ out) {
  __shared__ double sl[3 * kF64Plane], sr[3 * kF64Plane];
  const int tm = (int)blockIdx.x % ntile, tn = (int)blockIdx.x / ntile;
  const int nb = (ng + 15) / 16;
  const int ncol = HEAD ? 2 * nen : ng;
  // first block of the tile in both axes and its blocks, 1..4
  const int gb = tm * nb / ntile, hb = HEAD ? 4 * tn : tn * nb / ntile;
  const int nr = (tm + 1) * nb / ntile - gb;
  const int nc = HEAD ? min(4, (ncol + 15) / 16 - hb) : (tn + 1) * nb / ntile - hb;
  const int g0 = 16 * gb, h0 = 16 * hb;
  const int w = blockIdx.y, z = blockIdx.z;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int part = (wave + (int)(blockIdx.x + blockIdx.y + blockIdx.z)) & 3;
  const int li = lane & 15, lk = lane >> 4;
  const int hc = h0 + lane < ncol ? h0 + lane : ncol - 1;  // HEAD: this lane's column
  const double2* dww = dw + (size_t)(HEAD ? hc % nen : w) * ldd;
  const double dsgn = HEAD && hc >= nen ? -1.0 : 1.0;
  const size_t c0 = (size_t)z * chunks_per_split;
  const size_t c1 = c0 + chunks_per_split < nchunks ? c0 + chunks_per_split : nchunks;

  // thread (wave, lane) stages G = lane and G' = lane of the K rows wave and
  // wave + 4 of a chunk; the weight of a row is uniform in the wave
  constexpr int kE = kF64KC / 4;
  float2 la[kE], ra[kE];
  double2 dv[kE];
  auto load = [&](size_t c) {
#pragma unroll
    for (int e = 0; e < kE; ++e) {
      const size_t k = c * kF64KC + (size_t)(wave + 4 * e);
      la[e] = A[k * lda + g0 + lane];
      ra[e] = HEAD ? H[k] : A[k * lda + h0 + lane];
      dv[e] = dww[k];
      if (HEAD) dv[e].y *= dsgn;
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int e = 0; e < kE; ++e) {
      const int o = (wave + 4 * e) * kF64Row + lane;
      const double ar = la[e].x, ai = la[e].y;
      sl[o] = ar;
      sl[kF64Plane + o] = ai;
      sl[2 * kF64Plane + o] = ar + ai;
      const double cr = ra[e].x, ci = ra[e].y;
      const double br = dv[e].x * cr - dv[e].y * ci, bi = dv[e].x * ci + dv[e].y * cr;
      sr[o] = bi;
      sr[kF64Plane + o] = br;
      sr[2 * kF64Plane + o] = br + bi;
    }
  };

  d4v acc[3][4];
#pragma unroll
  for (int p = 0; p < 3; ++p)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[p][i] = d4v{0, 0, 0, 0};
  double2* o = out + ((size_t)z * (HEAD ? 1 : nen) + w) * (size_t)ng * ncol;
  // the chunk loop of a wave that owns NR x NC blocks from block (rb, cb) of
  // the tile on (none: it only stages)
  auto tile = [&](auto rows, auto cols, int rb, int cb) {
    constexpr int NR = decltype(rows)::value, NC = decltype(cols)::value;
    for (size_t c = c0; c < c1; ++c) {
      stage();
      __syncthreads();
      load(c + 1 < c1 ? c + 1 : c);
      if constexpr (NR > 0) f64_chunk<NR, NC>(sl + 16 * rb, sr + 16 * cb, li, lk, acc);
      __syncthreads();
    }
    // the FP64 MFMA leaves D[(lane>>4) + 4v][lane&15] in element v of a lane
#pragma unroll
    for (int a = 0; a < NR; ++a)
#pragma unroll
      for (int b = 0; b < NC; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int gi = g0 + (rb + a) * 16 + li;
          const int hj = h0 + (cb + b) * 16 + lk + 4 * v;
          const int i = a * NC + b;
          const double t1 = acc[0][i][v], t2 = acc[1][i][v], t3 = acc[2][i][v];
          if (gi < ng && hj < ncol) o[(size_t)hj * ng + gi] = make_double2(t3 - t1 - t2, t1 - t2);
        }
  };
  using std::integral_constant;
  const integral_constant<int, 0> n0{};
  const integral_constant<int, 1> n1{};
  const integral_constant<int, 2> n2{};
  const integral_constant<int, 3> n3{};
  if (c0 < c1) load(c0);
  if (nr == 4 && nc == 4) {
    tile(n2, n2, 2 * (part & 1), 2 * (part >> 1));
  } else if (nr == 2 && nc == 2) {
    tile(n1, n1, part & 1, part >> 1);
  } else if (nr <= nc) {  // a column of blocks per wave
    if (part >= nc) tile(n0, n0, 0, 0);
    else if (nr == 3) tile(n3, n1, 0, part);
    else if (nr == 2) tile(n2, n1, 0, part);
    else tile(n1, n1, 0, part);
  } else {  // a row of blocks per wave
    if (part >= nr) tile(n0, n0, 0, 0);
    else if (nc == 3) tile(n1, n3, part, 0);
    else if (nc == 2) tile(n1, n2, part, 0);
    else tile(n1, n1, part, 0);
  }
}

// chi[j] = sum_z partial[z][j] / volume, fixed order over z.
__global__ void k_chi_reduce(const double2* __restrict__ part, size_t n, int nsplit, double inv_vol,
                             double2* __restrict__ chi) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    double x = 0.0, y = 0.0;
    for (int z = 0; z < nsplit; ++z) {
      double2 v = part[(size_t)z * n + i];
      x += v.x;
      y += v.y;
    }
    chi[i] = make_double2(x * inv_vol, y * inv_vol);
  }
}

// chi of a further direction at q = 0: row and column g from its own partials
// (HEAD: k_chi_f64<true>'s [z][2][nen][ng], else tiles in chi's layout), every
// other element the first direction's (the same operands).
template <bool HEAD>
__global__ void k_chi_reduce_cross(const double2* __restrict__ part, int ng, int nen, int nsplit,
                                   double inv_vol, int g, const double2* __restrict__ chi0,
                                   double2* __restrict__ chi) {
  const size_t n = (size_t)ng * ng * nen, nh = 2 * (size_t)nen * ng;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const int gi = (int)(i % ng), hj = (int)(i / ng % ng);
    if (gi != g && hj != g) {
      chi[i] = chi0[i];
      continue;
    }
    const bool col = hj == g;
    const size_t w = i / ((size_t)ng * ng);
    const size_t at = HEAD ? (col ? w * ng + gi : (nen + w) * ng + hj) : i;
    double x = 0.0, y = 0.0;
    for (int z = 0; z < nsplit; ++z) {
      const double2 v = part[(size_t)z * (HEAD ? nh : n) + at];
      x += v.x;
      y += HEAD && !col ? -v.y : v.y;
    }
    chi[i] = make_double2(x * inv_vol, y * inv_vol);
  }
}

int chi_tile() { return kTile; }
int chi_kchunk() { return kKC; }

// K splits for 2048 workgroups: the fewest of either precision.
int chi_gemm_min_nsplit(int ng, int nen, size_t kpad) {
  const int ntile = (ng + kTile - 1) / kTile;
  const long wgs = (long)ntile * ntile * nen;
  return (int)std::min<long>((long)(kpad / kKC), (2048 + wgs - 1) / wgs);
}

// The most: 64, or twice the fewest where that is more, with partials of at most
// 2 GiB (one split whatever its size).
int chi_gemm_max_nsplit(int ng, int nen, size_t kpad) {
  const long room = (long)(2147483648.0 / (16.0 * ng * ng * nen));
  const long most = std::min(room, std::max(64L, 2L * chi_gemm_min_nsplit(ng, nen, kpad)));
  return (int)std::max(1L, std::min((long)(kpad / kKC), most));
}

// K splits.  FP32: the fewest.  FP64: at least as many, for the
// rounding of a sum falls with its splits (K 1296, NG 81: 9 splits left the real
// part off by 2.6e-16, 37 by 1.9e-16), and more where they are faster: with W workgroups per
// split, S = 4 resident per CU and C chunks of 32 K, a launch takes about
//   (W sp / S + 1/2 round of tail) (C / sp + 2 chunks of start and end)
// chunk times of a full CU (5.2 us: four workgroups' MFMAs), plus the traffic
// of the partial tiles, written and read once per split (32 bytes per element
// at about 4.5 TB/s); sp is where that is least.
int chi_gemm_nsplit(int prec, int ng, int nen, size_t kpad, int ncu) {
  const int fewest = chi_gemm_min_nsplit(ng, nen, kpad);
  if (prec != RP_PREC_FP64) return fewest;
  const int ntile = (ng + kTile - 1) / kTile;
  const double wgs = (double)ntile * ntile * nen;
  const double per = 16.0 * ng * ng * nen;  // bytes of one partial set
  const double cost = 2.0 * wgs / (4.0 * ncu) + 2.0 * per / 4.5e6 / 5.2;
  const double sp = std::min(64.0, std::round(std::sqrt(0.5 * (double)(kpad / kKC) / cost)));
  return std::min(std::max((int)sp, fewest), chi_gemm_max_nsplit(ng, nen, kpad));
}

void launch_chi_gemm(int prec, const float2* A, size_t lda, const double2* dw, size_t ldd,
                     size_t kpad, int ng, int nen, int nsplit, int cross, double2* partial,
                     hipStream_t s) {
  const int ntile = (ng + kTile - 1) / kTile;
  const size_t kchunks = kpad / kKC;
  const size_t per = (kchunks + nsplit - 1) / nsplit;
  dim3 grid(cross < 0 ? ntile * ntile : 2 * ntile - 1, nen, nsplit);
  constexpr size_t f = kKC / kF64KC;  // a split is a whole number of 32-row chunks in both
  switch (prec) {
    case RP_PREC_FP64:
      RP_CHECK(cross < 0, "k_chi_f64: row and column of one G are launch_chi_head's");
      hipLaunchKernelGGL(k_chi_f64<false>, grid, dim3(256), 0, s, A, lda, dw, ldd, per * f,
                         kchunks * f, ng, ntile, nen, (const float2*)nullptr, partial);
      break;
    case RP_PREC_FP32:
      hipLaunchKernelGGL(k_chi_gemm, grid, dim3(256), 0, s, A, lda, dw, ldd, per, kchunks, ng,
                         ntile, nen, cross < 0 ? -1 : cross / kTile, partial);
      break;
    default:
      throw Error("k_chi_gemm: FP64 or FP32 only (split-BF16 runs k_chi_bf16x3)");
  }
  RP_HIP(hipGetLastError());
}

// Zero fill by vector stores.  Used instead of hipMemsetAsync wherever the
// launch sequence may be captured into a graph (memset nodes are avoided there).
__global__ void k_zero(uint4* __restrict__ p, size_t n16, unsigned* __restrict__ tail,
                       size_t ntail) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride)
    p[i] = make_uint4(0u, 0u, 0u, 0u);
  if (blockIdx.x == 0 && threadIdx.x < ntail) tail[threadIdx.x] = 0u;
}

void launch_zero(void* p, size_t bytes, hipStream_t s) {
  if (bytes == 0) return;
  RP_CHECK(bytes % 4 == 0 && ((uintptr_t)p % 16) == 0, "zero fill needs 16-byte aligned words");
  const size_t n16 = bytes / 16, ntail = (bytes % 16) / 4;
  int blocks = (int)std::min<size_t>((n16 + 255) / 256, 4096);
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(k_zero, dim3(blocks), dim3(256), 0, s, (uint4*)p, n16,
                     (unsigned*)((char*)p + n16 * 16), ntail);
  RP_HIP(hipGetLastError());
}

void launch_chi_reduce_cross(const double2* partial, int ng, int nen, int nsplit, double inv_vol,
                             int g, const double2* chi0, double2* chi, hipStream_t s) {
  const unsigned blocks = (unsigned)std::min<size_t>(((size_t)ng * ng * nen + 255) / 256, 65536);
  hipLaunchKernelGGL(k_chi_reduce_cross<false>, dim3(blocks), dim3(256), 0, s, partial, ng, nen,
                     nsplit, inv_vol, g, chi0, chi);
  RP_HIP(hipGetLastError());
}

// One further direction at q = 0 in FP64 (its column g of A in place, H that
// column): row and column g, then the merge with the first direction's chi.
// room: double2 elements of partial.
void launch_chi_head(const float2* A, size_t lda, const double2* dw, size_t ldd, size_t kpad, int ng,
                     int nen, const float2* H, double inv_vol, int g, const double2* chi0,
                     double2* partial, size_t room, double2* chi, hipStream_t s) {
  const int ntile = (ng + kTile - 1) / kTile, ctile = (2 * nen + kTile - 1) / kTile;
  const size_t kchunks = kpad / kF64KC;
  // splits of at least 4 chunks (short sums round less), at most 64 of them, within the
  // partials' room
  size_t nsplit = std::min<size_t>(std::max<size_t>(1, kchunks / 4), 64);
  nsplit = std::min(nsplit, room / ((size_t)2 * nen * ng));
  RP_CHECK(nsplit >= 1, "chi head: no room for its partials");
  const size_t per = (kchunks + nsplit - 1) / nsplit;
  hipLaunchKernelGGL(k_chi_f64<true>, dim3(ntile * ctile, 1, (unsigned)nsplit), dim3(256), 0, s, A,
                     lda, dw, ldd, per, kchunks, ng, ntile, nen, H, partial);
  const unsigned blocks = (unsigned)std::min<size_t>(((size_t)ng * ng * nen + 255) / 256, 65536);
  hipLaunchKernelGGL(k_chi_reduce_cross<true>, dim3(blocks), dim3(256), 0, s, partial, ng, nen,
                     (int)nsplit, inv_vol, g, chi0, chi);
  RP_HIP(hipGetLastError());
}

void launch_chi_reduce(const double2* partial, size_t n, int nsplit, double inv_vol, double2* chi,
                       hipStream_t s) {
  int blocks = (int)((n + 255) / 256);
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(k_chi_reduce, dim3(blocks), dim3(256), 0, s, partial, n, nsplit, inv_vol, chi);
  RP_HIP(hipGetLastError());
}

}  // namespace rp
