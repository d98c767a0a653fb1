// calc_int (calc_w3d) on gfx950: the Wannier-basis bare and screened Coulomb
// integrals V_ij(R), W_ij(R,w) of calc_intW.F:636-985.
//
// rho_w(q+G) = (1/NTK) sum_k M_ww,k(G) / |q+G| comes from the pair-density
// kernels of rp_pairdens.hip (k_pair_kfft or k_pair_rsum, k_rho_from_grid: the products summed
// over k on the grid, one transform per (q, pair)).  Then per full-mesh q (all
// q of one launch):
//   func_ij(q)     = sum_{G in psi} rho_i(G) conj(rho_j(G))                (k_w_func)
//   funcw_ij(q,w)  = sum_{G,G' in eps} rho_i(G) eps^-1_q(G,G',w) conj(rho_j(G'))
//                    + sum_{G in psi \ eps} rho_i(G) conj(rho_j(G))        (k_w_contract)
// where eps^-1_q is the irreducible matrix (complex64, as the reference stores
// it) seen through the rotation of make_eps (calc_int_sub.F:222-311): an index
// map and a phase per G, folded into the rho vectors so that eps^-1 is read
// once, coalesced, straight from its irreducible copy.  Finally the lattice
// Fourier sums with the Hybertsen-Louie heads (k_w_fourier).
#include <algorithm>
#include <type_traits>

#include "rp_common.h"
#include "rp_kernels.h"

namespace rp {

// Per q: func (all G of the psi list) and the shell part of funcw (G beyond the
// eps sphere).  A wave per (q, i <= j), its lanes along G; (j, i) is the complex
// conjugate.  out [q][j][i].  64 q of five functions: 6 us, against 82 us of one
// workgroup per q that took the pairs in turn.
__global__ void __launch_bounds__(256) k_w_func(const double2* __restrict__ rho,
                                                const long long* __restrict__ rho_off,
                                                const int4* __restrict__ qinfo, int nwf, int ntq,
                                                double2* __restrict__ func,
                                                double2* __restrict__ shell) {
  const int np = nwf * (nwf + 1) / 2;
  const int u = (int)blockIdx.x * 4 + ((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (u >= ntq * np) return;  // uniform per wave
  const int q = u / np;
  int i = u % np, j = 0;
  while (i > j) i -= ++j;  // u % np = j (j + 1) / 2 + i, i <= j
  const int4 qi = qinfo[q];  // (ng_eps, ng_psi, iq_irr, trs)
  const int ngpsi = qi.y, nge = qi.x;
  const double2* ri = rho + rho_off[q] + (size_t)i * ngpsi;
  const double2* rj = rho + rho_off[q] + (size_t)j * ngpsi;
  double f[4] = {0, 0, 0, 0};  // func re/im, shell re/im
  for (int g = lane; g < ngpsi; g += 64) {
    const double2 a = ri[g], b = rj[g];
    const double pr = a.x * b.x + a.y * b.y, pi = a.y * b.x - a.x * b.y;  // a conj(b)
    f[0] += pr;
    f[1] += pi;
    if (g >= nge) { f[2] += pr; f[3] += pi; }
  }
#pragma unroll
  for (int c = 0; c < 4; ++c)
    for (int off = 32; off > 0; off >>= 1) f[c] += __shfl_xor(f[c], off);
  if (lane == 0) {
    const size_t ij = ((size_t)q * nwf + j) * nwf + i, ji = ((size_t)q * nwf + i) * nwf + j;
    func[ij] = make_double2(f[0], f[1]);
    shell[ij] = make_double2(f[2], f[3]);
    if (i != j) {
      func[ji] = make_double2(f[0], -f[1]);
      shell[ji] = make_double2(f[2], -f[3]);
    }
  }
}

// funcw for one w and a group of q that share one irreducible eps^-1 E
// (complex64, column-major): per member q, Y(a,c) = sum_b E(a,b) X_c(b), then
// funcw = sum_a Z(a) Y(a,.) + shell, where
//   trs = +1: X_j(b) = conj(rho_j(m^-1 b)) pf2, Z = rho_i(m^-1 a) pf1
//   trs = -1: X_i(b) = rho_i(m^-1 b) pf1,       Z = conj(rho_j(m^-1 a)) pf2
// with the member's own map m and phases.  The vectors are the NV <= 16 Wannier
// functions of calc_w3d per member, 16 / NV members per group at most, and
// every (i,j) of a member is formed, out [q][w][j][i] (calc_j3d's diagonal
// pairs: k_j_contract).  A workgroup takes all the vectors of its group, so E
// is read once per (group, w).  Y = E X runs on the FP64 matrix cores as in
// k_j_contract (Re Y = Er Xr - Ei Xi, Im Y = Er Xi + Ei Xr, v_mfma_f64_16x16x4,
// the group's vectors as one 16-column block): lane l supplies A(l % 16, l / 16)
// and B(l / 16, l % 16) and holds D(l / 16 + 4 v, l % 16).  X of every group
// is formed once (k_w_xvec, independent of w).  A wave takes up to kWA 16-row
// blocks of E per pass over all columns; then each lane multiplies its Y(a, c)
// by the Z_i(a) of c's member and keeps NV sums, reduced over the lanes of
// c and the waves at the end.
// Bound by the FP64 matrix cores, with 10 to 15 of the 16 columns in use: 64 q, 20
// frequencies, five functions, NG_eps ~ 310: 190 us with three row blocks per wave, 243
// with two, 218 with four; with the loads two steps ahead instead of one 212.  Three real
// products per complex one take 187 us, but Im Y = T3 - T1 - T2 left Im W of a diagonal
// pair 4 to 10 times further off by its own norm.
// grid: (nen, ngroups), 512 threads; group g has the q gmem[goff[g] .. goff[g+1]).
typedef double jd4 __attribute__((ext_vector_type(4)));
constexpr int kMaxWf = 16;     // Wannier functions of calc_w3d and calc_j3d
constexpr int kWcVec = 16;     // vectors of a group: one MFMA column block
constexpr int kWA = 3;         // row blocks per wave and pass of the W contraction
template <int NV>
constexpr int wc_members() { return kWcVec / NV; }
int w_contract_members(int nwf) { return kWcVec / nwf; }
int w_contract_vectors(int) { return kWcVec; }

// X_c(b) of every group, [nge][vb] at xw + vb * map_off[first member] (zero
// past the group's vectors).  grid: (ceil(largest nge / 16), ngroups), 256 threads.
__global__ void __launch_bounds__(256) k_w_xvec(const double2* __restrict__ rho,
                                                const long long* __restrict__ rho_off,
                                                const int4* __restrict__ qinfo,
                                                const int* __restrict__ minv,
                                                const double2* __restrict__ pf1,
                                                const double2* __restrict__ pf2,
                                                const long long* __restrict__ map_off,
                                                const int* __restrict__ goff,
                                                const int* __restrict__ gmem, int nv, int vb,
                                                double2* __restrict__ xw) {
  const int grp = blockIdx.y;
  const int mbeg = goff[grp], nvt = (goff[grp + 1] - mbeg) * nv;
  const int q0 = gmem[mbeg];
  const int nge = qinfo[q0].x;
  double2* out = xw + map_off[q0] * vb;
  const int e1 = min(vb * nge, ((int)blockIdx.x + 1) * 16 * vb);
  for (int e = (int)blockIdx.x * 16 * vb + (int)threadIdx.x; e < e1; e += blockDim.x) {
    const int b = e / vb, c = e % vb;
    double2 v = make_double2(0.0, 0.0);
    if (c < nvt) {
      const int q = gmem[mbeg + c / nv];
      const int4 qi = qinfo[q];
      const long long mo = map_off[q];
      const int g = minv[mo + b];
      const double2 rv = rho[rho_off[q] + (size_t)(c % nv) * qi.y + g];
      const double2 p = qi.w == 1 ? pf2[mo + g] : pf1[mo + g];
      // trs = +1: conj(rho) pf2; trs = -1: rho pf1
      const double xr = rv.x, xi = qi.w == 1 ? -rv.y : rv.y;
      v = make_double2(xr * p.x - xi * p.y, xr * p.y + xi * p.x);
    }
    out[e] = v;
  }
}

template <int NV>
__global__ void __launch_bounds__(512) k_w_contract(
    const float2* __restrict__ eps, const long long* __restrict__ eps_off,
    const double2* __restrict__ rho, const long long* __restrict__ rho_off,
    const int4* __restrict__ qinfo, const int* __restrict__ minv,
    const double2* __restrict__ pf1, const double2* __restrict__ pf2,
    const long long* __restrict__ map_off, const double2* __restrict__ shell,
    const int* __restrict__ goff, const int* __restrict__ gmem,
    const double2* __restrict__ xw, int nen, double2* __restrict__ funcw) {
  const int w = blockIdx.x, grp = blockIdx.y;
  const int mbeg = goff[grp], nm = goff[grp + 1] - mbeg;  // 1 <= nm <= 16 / NV
  const int nvt = nm * NV;
  const int q0m = gmem[mbeg];
  const int4 qi0 = qinfo[q0m];
  const int nge = qi0.x, iqir = qi0.z;
  const int ld = w3d_eps_ld(nge);
  const float2* E = eps + eps_off[iqir] + (size_t)w * ld * nge;
  const double2* Xg = xw + map_off[q0m] * kWcVec;  // (b, c) at Xg[b * 16 + c]
  __shared__ double red[kWcVec][NV][8][2];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int nab = (nge + 15) / 16;
  // this lane's vector c = li: member li / NV, its NV sums Z_i Y_c
  const bool cv = li < nvt;
  const int qm = gmem[mbeg + (cv ? li / NV : 0)];
  const int4 qim = qinfo[qm];
  const long long mom = map_off[qm];
  const double2* rm = rho + rho_off[qm];
  double sre[NV], sim[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) sre[i] = sim[i] = 0.0;
  // up to kWA row blocks per wave and pass (ab = a0 + wave + 8 j) share each
  // load of X; blocks past the last are skipped (uniform per wave)
  for (int a0 = 0; a0 < nab; a0 += 8 * kWA) {
    jd4 accr[kWA], acci[kWA];
    int arow[kWA];
#pragma unroll
    for (int j = 0; j < kWA; ++j) {
      accr[j] = acci[j] = jd4{0.0, 0.0, 0.0, 0.0};
      // rows nge .. ld-1 are the zero padding; their sums are never used
      arow[j] = (a0 + wave + 8 * j) * 16 + li;
    }
    const int nj = min(kWA, (nab - a0 - wave + 7) / 8);  // live blocks of this wave
    // X and E of the next step are loaded during a step's MFMAs; columns past nge
    // contribute zero
    double2 xq;
    float2 eq[kWA];
    auto fetch = [&](int b0) {
      const int b = min(b0 + lk, nge - 1);
      xq = Xg[(size_t)b * kWcVec + li];
#pragma unroll
      for (int j = 0; j < kWA; ++j) eq[j] = j < nj ? E[(size_t)b * ld + arow[j]] : make_float2(0.f, 0.f);
    };
    fetch(0);
    for (int b0 = 0; b0 < nge; b0 += 4) {
      const bool bv = b0 + lk < nge;
      const double xr = bv ? xq.x : 0.0, xi = bv ? xq.y : 0.0, nxi = -xi;
      double er[kWA], ei[kWA];
#pragma unroll
      for (int j = 0; j < kWA; ++j) {
        er[j] = eq[j].x;
        ei[j] = eq[j].y;
      }
      fetch(b0 + 4);
#pragma unroll
      for (int j = 0; j < kWA; ++j) {
        if (j >= nj) break;  // uniform
        accr[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(er[j], xr, accr[j], 0, 0, 0);
        acci[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(er[j], xi, acci[j], 0, 0, 0);
        accr[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ei[j], nxi, accr[j], 0, 0, 0);
        acci[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ei[j], xr, acci[j], 0, 0, 0);
      }
    }
    // Z_i(a) Y(a, c) for this lane's rows a = 16 ab + lk + 4 v and vector c = li
    if (cv) {
#pragma unroll
      for (int j = 0; j < kWA; ++j) {
        if (j >= nj) break;  // uniform
        const int ab = a0 + wave + 8 * j;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int ar = ab * 16 + lk + 4 * v;
          if (ar >= nge) continue;
          const int g = minv[mom + ar];
          const double yr = accr[j][v], yi = acci[j][v];
          const double2 pp = qim.w == 1 ? pf1[mom + g] : pf2[mom + g];
#pragma unroll
          for (int i = 0; i < NV; ++i) {
            const double2 rv = rm[(size_t)i * qim.y + g];
            double zr, zi;
            if (qim.w == 1) {  // Z = rho pf1
              zr = rv.x * pp.x - rv.y * pp.y;
              zi = rv.x * pp.y + rv.y * pp.x;
            } else {           // Z = conj(rho) pf2
              zr = rv.x * pp.x + rv.y * pp.y;
              zi = rv.x * pp.y - rv.y * pp.x;
            }
            sre[i] += zr * yr - zi * yi;
            sim[i] += zr * yi + zi * yr;
          }
        }
      }
    }
  }
  // lanes of one vector (li) hold their rows' sums: over lk, then the waves
#pragma unroll
  for (int i = 0; i < NV; ++i)
    for (int off = 16; off < 64; off <<= 1) {
      sre[i] += __shfl_xor(sre[i], off);
      sim[i] += __shfl_xor(sim[i], off);
    }
  if (lk == 0) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      red[li][i][wave][0] = sre[i];
      red[li][i][wave][1] = sim[i];
    }
  }
  __syncthreads();
  for (int e = t; e < 2 * nvt * NV; e += blockDim.x) {
    const int part = e & 1, idx = e >> 1;
    const int c = idx / NV, zi = idx % NV;
    const int m = c / NV, yc = c % NV;
    const int q = gmem[mbeg + m];
    // trs = +1 pairs Z_i Y_j, trs = -1 pairs Z_j Y_i
    const bool tp = qinfo[q].w == 1;
    const int i = tp ? zi : yc, j = tp ? yc : zi;
    double sum = 0.0;
#pragma unroll
    for (int wv = 0; wv < 8; ++wv) sum += red[c][zi][wv][part];
    const double2 sh = shell[((size_t)q * NV + j) * NV + i];
    double2* o = funcw + (((size_t)q * nen + w) * NV + j) * NV + i;
    if (part == 0) o->x = sum + sh.x;
    else o->y = sum + sh.y;
  }
}

// calc_j3d's contraction on the FP64 matrix cores: funcw_pp of the diagonal
// pairs of every R of a batch, by k_w_contract's formula.  A group is an
// irreducible q: its columns are the pair vectors of every full-mesh q that
// shares its eps^-1 and of every R, c = (member * nr + R) * npair + p, so that
// eps^-1 is read once per 64 columns instead of once per (q, R) and the columns
// fill the 16-wide blocks (25 pairs of one q and R fill 25 of 32; the 350 of two
// q and seven R all but two of 352).
//
// k_j_vecs forms once per batch, for every group, X [nbp][cpad] (nbp: NG_eps
// rounded up to 8 rows, cpad: the columns to 16, zero beyond) and Z [NG_eps][cpad].
// k_j_contract then takes 64 columns of one (group, w): Y = E X as real products
// (Re Y = Er Xr - Ei Xi, Im Y = Er Xi + Ei Xr) over tiles of up to 64 rows and 8
// columns of E at a time staged in LDS, and folds each tile into the sums over rows
// Z_c(a) Y(a, c).  A wave takes one column block of 16 and every row block of the
// tile (with fewer column blocks the rows are dealt out).  Bound by the FP64 MFMAs
// (shared with the FP64 vector unit, hence E and X widened once per workgroup): 64 q,
// 16 frequencies, 25 pairs, NG_eps ~310, seven R: 2.30 ms (59 TFLOP/s; 4.16 ms with
// every (q, R) on its own).  Four workgroups per CU; three take 2.41 ms; 12 columns of E
// at a time 2.55.  Three real products per complex one take 1.98 ms, but leave Im J
// further off (as Im W of k_w_contract).
constexpr int kJT = 64, kJKC = 8;                 // rows / columns of a tile, K per chunk
constexpr int kJRow = kJT + 16, kJPlane = kJKC * kJRow;

struct JGroup {
  int nge, iqir, mbeg, ncol;   // first member in gmem, columns
  long long xoff, zoff;        // first element of X and of Z
};

__global__ void __launch_bounds__(256) k_j_vecs(const double2* __restrict__ rho,
                                                const long long* __restrict__ rho_off,
                                                long long rho_r, const int4* __restrict__ qinfo,
                                                const int* __restrict__ minv,
                                                const double2* __restrict__ pf1,
                                                const double2* __restrict__ pf2,
                                                const long long* __restrict__ map_off,
                                                const JGroup* __restrict__ grp,
                                                const int* __restrict__ gmem, int np, int nr,
                                                double2* __restrict__ xs, double2* __restrict__ zs) {
  const JGroup g = grp[blockIdx.z];
  const int nbp = (g.nge + kJKC - 1) / kJKC * kJKC, cpad = (g.ncol + 15) / 16 * 16;
  const int c0 = blockIdx.x * 32, b0 = blockIdx.y * 32;
  if (c0 >= cpad || b0 >= nbp) return;
  __shared__ double2 sx[32][33], sz[32][33];  // [c][b]
  const int lane = threadIdx.x & 31, row = threadIdx.x >> 5;
  for (int i = row; i < 32; i += 8) {  // rows G along the lanes, one column each
    const int c = c0 + i, b = b0 + lane;
    double2 x = make_double2(0.0, 0.0), z = x;
    if (c < g.ncol && b < g.nge) {
      const int m = c / (nr * np), r = c / np % nr, p = c % np;
      const int q = gmem[g.mbeg + m];
      const int4 qi = qinfo[q];
      const long long mo = map_off[q];
      const int gg = minv[mo + b];
      const double2 v = rho[(long long)r * rho_r + rho_off[q] + (long long)p * qi.y + gg];
      const double2 p1 = pf1[mo + gg], p2 = pf2[mo + gg];
      // trs = +1: X = conj(rho) pf2, Z = rho pf1; trs = -1: X = rho pf1, Z = conj(rho) pf2
      const double2 a = make_double2(v.x * p1.x - v.y * p1.y, v.x * p1.y + v.y * p1.x);
      const double2 d = make_double2(v.x * p2.x + v.y * p2.y, v.x * p2.y - v.y * p2.x);
      x = qi.w == 1 ? d : a;
      z = qi.w == 1 ? a : d;
    }
    sx[i][lane] = x;
    sz[i][lane] = z;
  }
  __syncthreads();
  for (int i = row; i < 32; i += 8) {  // columns along the lanes
    const int b = b0 + i, c = c0 + lane;
    if (b >= nbp || c >= cpad) continue;
    const double2 x = sx[lane][i];
    xs[g.xoff + (size_t)b * cpad + c] = x;
    if (b < g.nge) zs[g.zoff + (size_t)b * cpad + c] = sz[lane][i];
  }
}

// NR row blocks from block rb on by the column block cb of a staged chunk.  (Unrolled, the
// loop's operands do not fit beside the sums in the 128 registers of four workgroups.)
template <int NR>
__device__ __forceinline__ void j_chunk(const double* pe, const double* px, int rb, int cb, int li,
                                        int lk, jd4 (&re)[NR], jd4 (&im)[NR]) {
#pragma unroll 1
  for (int k0 = 0; k0 < kJKC; k0 += 4) {
    const int o = (k0 + lk) * kJRow + li;
    const double xr = px[o + 16 * cb], xi = px[kJPlane + o + 16 * cb], nxi = -xi;
    double er[NR], ei[NR];
#pragma unroll
    for (int a = 0; a < NR; ++a) {
      er[a] = pe[o + 16 * (rb + a)];
      ei[a] = pe[kJPlane + o + 16 * (rb + a)];
    }
#pragma unroll
    for (int a = 0; a < NR; ++a) {
      re[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(er[a], xr, re[a], 0, 0, 0);
      im[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(er[a], xi, im[a], 0, 0, 0);
    }
#pragma unroll
    for (int a = 0; a < NR; ++a) {
      re[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(ei[a], nxi, re[a], 0, 0, 0);
      im[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(ei[a], xr, im[a], 0, 0, 0);
    }
  }
}

// grid: (nen, groups, column tiles of the widest group x nrs), 256 threads; row
// tile t of a workgroup with row share s (of nrs) is taken when t % nrs == s.
// out[s][R][q][w][p]: the partial sums over that share's rows.
__global__ void __launch_bounds__(256, 4) k_j_contract(
    const float2* __restrict__ eps, const long long* __restrict__ eps_off,
    const JGroup* __restrict__ grp, const int* __restrict__ gmem, const double2* __restrict__ xs,
    const double2* __restrict__ zs, int np, int nr, int nrs, int ntq, int nen,
    double2* __restrict__ out) {
  __shared__ double se[2 * kJPlane], sx[2 * kJPlane];
  __shared__ double2 red[4][16];
  __shared__ double2 sum[256];  // each thread's rows of its column so far (not in registers
                                // through the loops over b)
  const int w = blockIdx.x, rs = (int)blockIdx.z % nrs, tc = (int)blockIdx.z / nrs;
  const JGroup g = grp[blockIdx.y];
  const int ncb = (g.ncol + 15) / 16, nct = (ncb + 3) / 4, cpad = 16 * ncb;
  if (tc >= nct) return;  // uniform
  const int hb = tc * ncb / nct, nc = (tc + 1) * ncb / nct - hb;  // column blocks, dealt evenly
  const int nab = (g.nge + 15) / 16, nat = (nab + 3) / 4;
  const int ld = w3d_eps_ld(g.nge), nbp = (g.nge + kJKC - 1) / kJKC * kJKC;
  const float2* E = eps + eps_off[g.iqir] + (size_t)w * ld * g.nge;
  const double2* X = xs + g.xoff;
  const double2* Z = zs + g.zoff;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int part = (wave + (int)(blockIdx.x + blockIdx.y)) & 3;
  const int li = lane & 15, lk = lane >> 4;
  // this wave's column block and share of a tile's row blocks
  const int cb = nc >= 3 ? part : (nc == 2 ? part & 1 : 0);
  const int nsh = nc >= 3 ? 1 : (nc == 2 ? 2 : 4), sh = nc >= 3 ? 0 : (nc == 2 ? part >> 1 : part);
  const int xc = min(16 * hb + lane, cpad - 1);
  float2 ev[kJKC / 4];
  double2 xv[kJKC / 4];
  auto load = [&](int a0, int b0) {
    const int a = min(a0 + lane, ld - 1);
#pragma unroll
    for (int e = 0; e < kJKC / 4; ++e) {
      const int b = b0 + wave + 4 * e;
      ev[e] = (E + (size_t)min(b, g.nge - 1) * ld)[a];  // X is zero past NG_eps
      xv[e] = (X + (size_t)b * cpad)[xc];
    }
  };
  sum[threadIdx.x] = make_double2(0.0, 0.0);
  if (rs < nat) load(16 * (rs * nab / nat), 0);
  // one row tile for a wave with NR of its row blocks, from rb on (0: it only
  // stages); next: first row of the workgroup's next tile, < 0 for none
  auto tile = [&](auto rows, int ab, int rb, int next) {
    constexpr int NR = decltype(rows)::value;
    jd4 re[NR > 0 ? NR : 1], im[NR > 0 ? NR : 1];
#pragma unroll
    for (int a = 0; a < NR; ++a) re[a] = im[a] = jd4{0, 0, 0, 0};
    for (int b0 = 0; b0 < nbp; b0 += kJKC) {
#pragma unroll
      for (int e = 0; e < kJKC / 4; ++e) {
        const int o = (wave + 4 * e) * kJRow + lane;
        se[o] = ev[e].x;
        se[kJPlane + o] = ev[e].y;
        sx[o] = xv[e].x;
        sx[kJPlane + o] = xv[e].y;
      }
      __syncthreads();
      if (b0 + kJKC < nbp) load(16 * ab, b0 + kJKC);
      else if (next >= 0) load(next, 0);
      if constexpr (NR > 0) j_chunk<NR>(se, sx, rb, cb, li, lk, re, im);
      __syncthreads();
    }
    // (the compiler would form every row's and the column's index before the loop over
    // b and keep them in registers through it)
    int row = lk, col = li;
    asm volatile("" : "+v"(row), "+v"(col));
    const int c = 16 * (hb + cb) + col;
    double sre = sum[threadIdx.x].x, sim = sum[threadIdx.x].y;
#pragma unroll
    for (int a = 0; a < NR; ++a) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int ar = 16 * (ab + rb + a) + row + 4 * v;
        if (ar >= g.nge) continue;
        const double yr = re[a][v], yi = im[a][v];
        const double2 z = Z[(size_t)ar * cpad + c];
        sre += z.x * yr - z.y * yi;
        sim += z.x * yi + z.y * yr;
        if (v & 1) __builtin_amdgcn_sched_barrier(0);  // few Z in registers at a time: no spills
      }
    }
    sum[threadIdx.x] = make_double2(sre, sim);
  };
  using std::integral_constant;
  for (int t = rs; t < nat; t += nrs) {
    const int ab = t * nab / nat, na = (t + 1) * nab / nat - ab;
    const int rb = na * sh / nsh, nrb = cb < nc ? na * (sh + 1) / nsh - rb : 0;
    const int next = t + nrs < nat ? 16 * ((t + nrs) * nab / nat) : -1;
    if (nrb == 4) tile(integral_constant<int, 4>{}, ab, rb, next);
    else if (nrb == 3) tile(integral_constant<int, 3>{}, ab, rb, next);
    else if (nrb == 2) tile(integral_constant<int, 2>{}, ab, rb, next);
    else if (nrb == 1) tile(integral_constant<int, 1>{}, ab, rb, next);
    else tile(integral_constant<int, 0>{}, ab, rb, next);
  }
  double sre = sum[threadIdx.x].x, sim = sum[threadIdx.x].y;
  for (int off = 16; off < 64; off <<= 1) {
    sre += __shfl_xor(sre, off);
    sim += __shfl_xor(sim, off);
  }
  if (lk == 0) red[part][li] = make_double2(sre, sim);
  __syncthreads();
  for (int e = threadIdx.x; e < 16 * nc; e += 256) {
    const int k = e / 16, c = 16 * (hb + k) + e % 16;
    if (c >= g.ncol) continue;
    double2 v = red[k][e % 16];  // the shares of column block k: parts k, k + 4 / nsh, ...
    for (int i = 1; i < nsh; ++i) {
      const double2 u = red[k + i * (4 / nsh)][e % 16];
      v.x += u.x;
      v.y += u.y;
    }
    const int m = c / (nr * np), r = c / np % nr, p = c % np;
    const int q = gmem[g.mbeg + m];
    out[((((size_t)rs * nr + r) * ntq + q) * nen + w) * np + p] = v;
  }
}

// calc_j3d func / shell (calc_intJ.F:680-690): per (R, q, p) sum_G |rho_p(G)|^2
// (real) over every G and over the shell beyond the eps sphere.  A wave per
// (R, q, p); out [R][q][p] as (all, shell).
__global__ void __launch_bounds__(256) k_j_func(const double2* __restrict__ rho,
                                                const long long* __restrict__ rho_off,
                                                long long rho_r, const int4* __restrict__ qinfo,
                                                int np, int ntq, int nr,
                                                double2* __restrict__ func) {
  const int u = (int)blockIdx.x * 4 + ((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (u >= nr * ntq * np) return;  // uniform per wave
  const int p = u % np, q = u / np % ntq, r = u / (np * ntq);
  const int4 qi = qinfo[q];
  const double2* v = rho + (long long)r * rho_r + rho_off[q] + (long long)p * qi.y;
  double f = 0.0, sh = 0.0;
  for (int g = lane; g < qi.y; g += 64) {
    const double2 a = v[g];
    const double m = a.x * a.x + a.y * a.y;
    f += m;
    if (g >= qi.x) sh += m;
  }
  for (int off = 32; off > 0; off >>= 1) {
    f += __shfl_xor(f, off);
    sh += __shfl_xor(sh, off);
  }
  if (lane == 0) func[u] = make_double2(f, sh);
}

// X_ij(R) (slot w = nen) and J_ij(R, w) = 2*2pi sum_q f(q) / V / NTQ, heads on
// i = j at R = 0 (calc_intJ.F:830-904); f(q) is func, or the contraction's row
// shares plus the shell.  grid (nen + 1, R of the batch), 256 threads: the q are
// dealt to nq threads per pair and their sums meet in LDS, pair by pair in turn.
// out: X [p] and J [w * wstride + p] at each R's slot.
__global__ void __launch_bounds__(256) k_j_sum(const double2* __restrict__ func,
                                               const double2* __restrict__ funcw, int ntq, int nwf,
                                               int nen, int nr, int nrs,
                                               const int* __restrict__ isr0, double volume,
                                               double chead, const double2* __restrict__ cheadw,
                                               double2* __restrict__ xmat,
                                               double2* __restrict__ jmat, size_t wstride) {
  const int w = blockIdx.x, r = blockIdx.y, np = nwf * nwf;
  const bool isx = w == nen;
  const double tpi = 2.0 * 3.141592653589793238462643383279502884;
  __shared__ double2 red[256];
  const int pb = np < 256 ? np : 256, nq = 256 / pb;  // pairs at a time, threads per pair
  for (int p0 = 0; p0 < np; p0 += pb) {
    const int p = p0 + (int)threadIdx.x % pb, ql = (int)threadIdx.x / pb;
    double sr = 0.0, si = 0.0;
    if (ql < nq && p < np)
      for (int q = ql; q < ntq; q += nq) {
        const double2 f = func[((size_t)r * ntq + q) * np + p];
        if (isx) {
          sr += f.x;
        } else {
          sr += f.y;
          for (int s = 0; s < nrs; ++s) {
            const double2 v = funcw[((((size_t)s * nr + r) * ntq + q) * nen + w) * np + p];
            sr += v.x;
            si += v.y;
          }
        }
      }
    __syncthreads();
    red[threadIdx.x] = make_double2(sr, si);
    __syncthreads();
    if (ql == 0 && p < np) {
      for (int k = 1; k < nq; ++k) {
        sr += red[threadIdx.x + k * pb].x;
        si += red[threadIdx.x + k * pb].y;
      }
      double xr = 2.0 * tpi * sr / volume / (double)ntq, xi = 2.0 * tpi * si / volume / (double)ntq;
      const bool diag = isr0[r] && (p % nwf) == (p / nwf);
      if (isx) {
        if (diag) xr += chead;
        xmat[(size_t)r * np + p] = make_double2(xr, xi);
      } else {
        if (diag) { xr += cheadw[w].x; xi += cheadw[w].y; }
        jmat[(size_t)w * wstride + (size_t)r * np + p] = make_double2(xr, xi);
      }
    }
  }
}

// V_ij(R) (slot w = nen) and W_ij(R,w): 2*2pi sum_q f_ij(q) e^{-i 2pi q.R} / V / NTQ
// + head (calc_intW.F:942-985).  grid: (nR, nen + 1), 64 threads, up to four
// (i,j) each (NWF <= 16); the phases of a block's R are formed once per q in
// LDS.  out: V [R][j][i], W [w][R][j][i].
__global__ void __launch_bounds__(64) k_w_fourier(const double2* __restrict__ func,
                                                  const double2* __restrict__ funcw,
                                                  const double* __restrict__ sq, int ntq, int nwf,
                                                  int nen, int na1, int na2, int na3,
                                                  double volume, double chead,
                                                  const double2* __restrict__ cheadw,
                                                  double2* __restrict__ vmat,
                                                  double2* __restrict__ wmat) {
  const int r = blockIdx.x, w = blockIdx.y;
  const int n1 = 2 * na1 + 1, n2 = 2 * na2 + 1;
  const int ia1 = r % n1 - na1, ia2 = (r / n1) % n2 - na2, ia3 = r / (n1 * n2) - na3;
  const double tpi = 2.0 * 3.141592653589793238462643383279502884;
  const bool isv = w == nen;
  const int np = nwf * nwf;  // <= 256: four (i, j) per thread
  // e^{-i phase(q)} of kWfQ q at a time in LDS, shared by every (i, j)
  constexpr int kWfQ = 256;
  __shared__ double2 ph[kWfQ];
  double sr[4] = {0.0, 0.0, 0.0, 0.0}, si[4] = {0.0, 0.0, 0.0, 0.0};
  for (int qb = 0; qb < ntq; qb += kWfQ) {
    const int nq = min(kWfQ, ntq - qb);
    __syncthreads();
    for (int e = threadIdx.x; e < nq; e += blockDim.x) {
      const int q = qb + e;
      const double phase = tpi * (sq[3 * q] * (double)ia1 + sq[3 * q + 1] * (double)ia2 +
                                  sq[3 * q + 2] * (double)ia3);
      double sn, cs;
      sincos(phase, &sn, &cs);
      ph[e] = make_double2(cs, sn);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int ij = threadIdx.x + 64 * u;
      if (ij >= np) break;
      const int i = ij % nwf, j = ij / nwf;
      for (int e = 0; e < nq; ++e) {
        const int q = qb + e;
        const double2 f = isv ? func[((size_t)q * nwf + j) * nwf + i]
                              : funcw[(((size_t)q * nen + w) * nwf + j) * nwf + i];
        const double c = ph[e].x, sn = ph[e].y;
        // f * exp(-i phase)
        sr[u] += f.x * c + f.y * sn;
        si[u] += f.y * c - f.x * sn;
      }
    }
  }
  const double sc = 2.0 * tpi;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int ij = threadIdx.x + 64 * u;
    if (ij >= np) break;
    const int i = ij % nwf, j = ij / nwf;
    if (isv) {
      vmat[((size_t)r * nwf + j) * nwf + i] = make_double2(
          sc * sr[u] / volume / (double)ntq + chead, sc * si[u] / volume / (double)ntq);
    } else {
      const double2 h = cheadw[w];
      wmat[(((size_t)w * (n1 * n2 * (2 * na3 + 1)) + r) * nwf + j) * nwf + i] =
          make_double2(sc * sr[u] / volume / (double)ntq + h.x, sc * si[u] / volume / (double)ntq + h.y);
    }
  }
}

int w3d_max_wannier() { return kMaxWf; }

void launch_w_func(const double2* rho, const long long* rho_off, const int4* qinfo, int ntq,
                   int nwf, double2* func, double2* shell, hipStream_t s) {
  const int units = ntq * (nwf * (nwf + 1) / 2);
  hipLaunchKernelGGL(k_w_func, dim3((units + 3) / 4), dim3(256), 0, s, rho, rho_off, qinfo, nwf, ntq, func,
                     shell);
  RP_HIP(hipGetLastError());
}

void launch_w_contract(const float2* eps, const long long* eps_off, const double2* rho,
                       const long long* rho_off, const int4* qinfo, const int* minv,
                       const double2* pf1, const double2* pf2, const long long* map_off,
                       const double2* shell, const int* goff, const int* gmem, int ngroups,
                       int nwf, int nen, int max_nge, double2* xw, double2* funcw,
                       hipStream_t s) {
  RP_CHECK(nwf >= 1 && nwf <= kMaxWf, "W contraction supports 1..16 Wannier functions");
  RP_CHECK(max_nge >= 1, "W contraction: empty eps sphere");
  if (ngroups <= 0) return;
  hipLaunchKernelGGL(k_w_xvec, dim3((max_nge + 15) / 16, ngroups), dim3(256), 0, s, rho, rho_off, qinfo, minv, pf1,
                     pf2, map_off, goff, gmem, nwf, w_contract_vectors(nwf), xw);
  switch (nwf) {
#define RP_WC(NV)                                                                             \
  case NV:                                                                                    \
    hipLaunchKernelGGL((k_w_contract<NV>), dim3(nen, ngroups), dim3(512), 0, s, eps, eps_off, \
                       rho, rho_off, qinfo, minv, pf1, pf2, map_off, shell, goff, gmem, xw,   \
                       nen, funcw);                                                           \
    break;
    RP_WC(1) RP_WC(2) RP_WC(3) RP_WC(4) RP_WC(5) RP_WC(6) RP_WC(7) RP_WC(8)
    RP_WC(9) RP_WC(10) RP_WC(11) RP_WC(12) RP_WC(13) RP_WC(14) RP_WC(15) RP_WC(16)
#undef RP_WC
  }
  RP_HIP(hipGetLastError());
}

// Elements of X and of Z that a group of nge rows and ncol columns takes.
size_t j_x_elems(int nge, int ncol) {
  return (size_t)((nge + kJKC - 1) / kJKC * kJKC) * ((ncol + 15) / 16 * 16);
}
size_t j_z_elems(int nge, int ncol) { return (size_t)nge * ((ncol + 15) / 16 * 16); }

// Shares of the row tiles (1..4): workgroups for a few rounds of four per CU.
int j_row_shares(int ngroups, int nen, int max_ncol, int max_nge, int ncu) {
  const long wgs = (long)ngroups * nen * ((max_ncol + kJT - 1) / kJT);
  const int nat = (max_nge + kJT - 1) / kJT;
  const long want = (4L * 4 * ncu + wgs - 1) / std::max(1L, wgs);
  return (int)std::min<long>(std::min(4, nat), std::max(1L, want));
}

// groups: device array of ngroups {nge, iq_irr, first member, columns, X offset,
// Z offset} as pack_j_group lays them out; nr R of the batch, rho_r apart.
size_t j_group_bytes() { return sizeof(JGroup); }
void pack_j_group(void* at, int nge, int iqir, int mbeg, int ncol, long long xoff, long long zoff) {
  *(JGroup*)at = JGroup{nge, iqir, mbeg, ncol, xoff, zoff};
}

void launch_j_contract(const float2* eps, const long long* eps_off, const double2* rho,
                       const long long* rho_off, long long rho_r, const int4* qinfo,
                       const int* minv, const double2* pf1, const double2* pf2,
                       const long long* map_off, const void* groups, const int* gmem, int ngroups,
                       int max_nge, int max_ncol, int npair, int nr, int nrs, int ntq, int nen,
                       double2* xs, double2* zs, double2* funcw, hipStream_t s) {
  RP_CHECK(ngroups >= 1 && ngroups <= 65535 && max_nge >= 1 && max_ncol >= 1,
           "J contraction: bad group sizes");
  const int cpad = (max_ncol + 15) / 16 * 16, nbp = (max_nge + kJKC - 1) / kJKC * kJKC;
  hipLaunchKernelGGL(k_j_vecs, dim3((cpad + 31) / 32, (nbp + 31) / 32, ngroups), dim3(256), 0, s, rho,
                     rho_off, rho_r, qinfo, minv, pf1, pf2, map_off, (const JGroup*)groups, gmem,
                     npair, nr, xs, zs);
  hipLaunchKernelGGL(k_j_contract, dim3(nen, ngroups, (cpad + kJT - 1) / kJT * nrs), dim3(256), 0, s,
                     eps, eps_off, (const JGroup*)groups, gmem, (const double2*)xs,
                     (const double2*)zs, npair, nr, nrs, ntq, nen, funcw);
  RP_HIP(hipGetLastError());
}

void launch_j_func(const double2* rho, const long long* rho_off, long long rho_r, const int4* qinfo,
                   int ntq, int npair, int nr, double2* func, hipStream_t s) {
  const long units = (long)nr * ntq * npair;
  hipLaunchKernelGGL(k_j_func, dim3((unsigned)((units + 3) / 4)), dim3(256), 0, s, rho, rho_off, rho_r,
                     qinfo, npair, ntq, nr, func);
  RP_HIP(hipGetLastError());
}

void launch_j_sum(const double2* func, const double2* funcw, int ntq, int nwf, int nen, int nr, int nrs,
                  const int* isr0, double volume, double chead, const double2* cheadw, double2* xmat,
                  double2* jmat, size_t wstride, hipStream_t s) {
  hipLaunchKernelGGL(k_j_sum, dim3(nen + 1, nr), dim3(256), 0, s, func, funcw, ntq, nwf, nen, nr, nrs,
                     isr0, volume, chead, cheadw, xmat, jmat, wstride);
  RP_HIP(hipGetLastError());
}

void launch_w_fourier(const double2* func, const double2* funcw, const double* sq, int ntq, int nwf,
                      int nen, const int na[3], double volume, double chead, const double2* cheadw,
                      double2* vmat, double2* wmat, hipStream_t s) {
  const int nr = (2 * na[0] + 1) * (2 * na[1] + 1) * (2 * na[2] + 1);
  hipLaunchKernelGGL(k_w_fourier, dim3(nr, nen + 1), dim3(64), 0, s, func, funcw, sq, ntq, nwf,
                     nen, na[0], na[1], na[2], volume, chead, cheadw, vmat, wmat);
  RP_HIP(hipGetLastError());
}

}  // namespace rp
