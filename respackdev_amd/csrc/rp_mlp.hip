// Band-tail closure network on gfx950: a small MLP (fully connected layers,
// GELU on the hidden layers, linear output) with BF16 weights and FP32
// activations and accumulation, and its training (mean-squared error, Adam on
// FP32 master weights).
//
// Layout: activations [n][width] row-major FP32; weights W_l [out][in] BF16
// (converted from the FP32 masters before each forward pass); biases FP32.
//   forward : Z_l = A_{l-1} W_l^T + b_l,  A_l = gelu(Z_l) (hidden), Y = Z_L
//   backward: dW_l = dZ_l^T A_{l-1},  db_l = sum_n dZ_l,
//             dA_{l-1} = dZ_l W_l,  dZ_{l-1} = dA_{l-1} * gelu'(Z_{l-1})
// The weight gradient is reduced over samples in fixed chunks (partial sums,
// then a reduction kernel) so results do not depend on launch timing.
#include <algorithm>

#include "rp_common.h"
#include "rp_kernels.h"

namespace rp {

namespace {
constexpr int kRows = 32;      // samples per forward / data-gradient block
constexpr int kMaxIn = 128;    // widest layer input
constexpr int kChunk = 256;    // samples per weight-gradient partial
}  // namespace

__device__ __forceinline__ float bf16_round_to_float(unsigned short h) {
  return __builtin_bit_cast(float, (unsigned)h << 16);
}

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float x) {
  const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
  const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
  return cdf + x * pdf;
}

// FP32 master -> BF16 (round to nearest even), n values.
__global__ void k_to_bf16(const float* __restrict__ src, size_t n, unsigned short* __restrict__ dst) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    __bf16 h = (__bf16)src[i];
    dst[i] = __builtin_bit_cast(unsigned short, h);
  }
}

// Layers whose input width K is 8, 16, 32, 64 or 128 and whose output is at
// least 16 wide (the closure's hidden layers).  A workgroup holds W in LDS as
// pairs of BF16 inputs [K/2][cols], a wave takes 64 outputs of 8 samples: lane c
// reads its pair of weights once for the eight samples, whose inputs are uniform
// over the wave and arrive through scalar loads, 8 inputs at a time.  The loop
// over the inputs stays rolled: unrolled, the compiler issues every scalar load
// at its start and spills.  Each output sums b + a_0 w_0 + a_1 w_1 + ... in that
// order, as k_linear_fwd does: the same bits.  Bound by the FP32 FMAs and the
// scalar loads' latency: 60000 samples of 128 -> 128 take 47 us (42 TFLOP/s), and
// a forward pass of 300011 samples 1.23 ms with its copies, against 3.03 ms when
// every layer ran k_linear_fwd (W read uncoalesced, once per sample).  Z, A:
// pre-activation and gelu(Z), each optional.  Rows up to a multiple of kRowsS past n are read (in is
// allocated for them), their results are not stored.
constexpr int kRowsS = 8;     // samples per wave at most
// Batches from here on take 8 samples per wave; smaller ones 4, which gives the
// scalar loads' latency two waves per SIMD at 4096 samples (a 128 -> 128 layer
// 13.1 us with 8, 9.4 us with 4 and rows_touch).
constexpr int kRowsBig = 16384;
template <int K, int S>
__device__ __forceinline__ void rows_loop(const float* __restrict__ row,
                                          const unsigned (*sw)[kMaxIn + 1], int cl,
                                          float (&acc)[S]) {
  constexpr int CH = K < 64 / S ? K : 64 / S;  // inputs per pass: 64 scalar registers
#pragma unroll 1
  for (int j = 0; j < K; j += CH) {
#pragma unroll
    for (int e = 0; e < CH; e += 2) {
      const unsigned u = sw[(j + e) / 2][cl];
      const float w0 = __builtin_bit_cast(float, u << 16);
      const float w1 = __builtin_bit_cast(float, u & 0xffff0000u);
#pragma unroll
      for (int s = 0; s < S; ++s)
        acc[s] = fmaf(row[s * K + j + e + 1], w1, fmaf(row[s * K + j + e], w0, acc[s]));
    }
  }
}

// One load of every 64-byte line of S rows of K floats, so that the scalar loads
// that follow find them in this XCD's L2 (the rows come from other XCDs).
template <int K, int S>
__device__ __forceinline__ void rows_touch(const float* __restrict__ row, int lane) {
  constexpr int lines = (S * K + 15) / 16;
  const float v = row[16 * (lane < lines ? lane : 0)];
  asm volatile("" ::"v"(v));
}

template <int K, int S>
__global__ void __launch_bounds__(256) k_rows_fwd(const float* __restrict__ in, int n,
                                                  const unsigned short* __restrict__ W,
                                                  const float* __restrict__ b, int cols,
                                                  float* __restrict__ Z, float* __restrict__ Aout) {
  __shared__ unsigned sw[K / 2][kMaxIn + 1];  // + 1: the staging writes fall on different banks
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int cw = (cols + 63) / 64;  // 1 or 2
  int r0 = ((int)blockIdx.x * (4 / cw) + wave / cw) * S;
  if (r0 < n) rows_touch<K, S>(in + (size_t)r0 * K, lane);
  for (int e = threadIdx.x; e < cols * (K / 8); e += 256) {
    const int c = e / (K / 8), j = e % (K / 8);
    const uint4 v = ((const uint4*)W)[e];
    sw[4 * j][c] = v.x;
    sw[4 * j + 1][c] = v.y;
    sw[4 * j + 2][c] = v.z;
    sw[4 * j + 3][c] = v.w;
  }
  __syncthreads();
  const int c = (wave % cw) * 64 + lane, cl = c < cols ? c : cols - 1;
  const float bias = b[cl];
  const int step = (int)gridDim.x * (4 / cw) * S;
  for (; r0 < n; r0 += step) {
    if (r0 + step < n) rows_touch<K, S>(in + (size_t)(r0 + step) * K, lane);
    float acc[S];
#pragma unroll
    for (int s = 0; s < S; ++s) acc[s] = bias;
    rows_loop<K, S>(in + (size_t)r0 * K, sw, cl, acc);
    if (c < cols) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        if (r0 + s >= n) break;
        const size_t idx = (size_t)(r0 + s) * cols + c;
        if (Z) Z[idx] = acc[s];
        if (Aout) Aout[idx] = gelu(acc[s]);
      }
    }
  }
}

// Narrow outputs (fewer than 16: the last layer): a thread per sample, W uniform
// over the wave; nin a multiple of 4.  The same sums as k_linear_fwd.  With
// targets T also the mean-squared error, as k_mse: dY = 2 (Y - T) scale and the
// block's loss sum.
__global__ void __launch_bounds__(64) k_narrow_fwd(const float* __restrict__ in, int n, int nin,
                                                   const unsigned short* __restrict__ W,
                                                   const float* __restrict__ b, int nout, int act,
                                                   float* __restrict__ Z, float* __restrict__ Aout,
                                                   const float* __restrict__ T, float scale,
                                                   float* __restrict__ dY, double* __restrict__ lossp) {
  const int r = blockIdx.x * 64 + threadIdx.x;
  const float4* row = (const float4*)(in + (size_t)(r < n ? r : 0) * nin);
  double loss = 0.0;
  for (int o = 0; o < nout && r < n; ++o) {
    const unsigned short* w = W + (size_t)o * nin;
    float acc = b[o];
#pragma unroll 8
    for (int j = 0; j < nin / 4; ++j) {
      const float4 x = row[j];
      acc = fmaf(x.x, bf16_round_to_float(w[4 * j]), acc);
      acc = fmaf(x.y, bf16_round_to_float(w[4 * j + 1]), acc);
      acc = fmaf(x.z, bf16_round_to_float(w[4 * j + 2]), acc);
      acc = fmaf(x.w, bf16_round_to_float(w[4 * j + 3]), acc);
    }
    const size_t idx = (size_t)r * nout + o;
    if (Z) Z[idx] = acc;
    if (act) Aout[idx] = gelu(acc);
    if (T) {
      const float d = acc - T[idx];
      dY[idx] = 2.0f * d * scale;
      loss += (double)d * d;
    }
  }
  if (T) {  // uniform
    for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off);
    if (threadIdx.x == 0) lossp[blockIdx.x] = loss;
  }
}

// Any other width: Z = A W^T + b over a block of kRows samples; A_out = gelu(Z) when act.
// grid: ceil(n / kRows); block 256.  nin <= kMaxIn.
__global__ void __launch_bounds__(256) k_linear_fwd(const float* __restrict__ A, int n, int nin,
                                                   const unsigned short* __restrict__ W,
                                                   const float* __restrict__ b, int nout, int act,
                                                   float* __restrict__ Z, float* __restrict__ Aout) {
  __shared__ float sA[kRows][kMaxIn + 1];
  const int r0 = blockIdx.x * kRows;
  for (int e = threadIdx.x; e < kRows * nin; e += blockDim.x) {
    const int r = e / nin, i = e % nin;
    sA[r][i] = r0 + r < n ? A[(size_t)(r0 + r) * nin + i] : 0.0f;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kRows * nout; e += blockDim.x) {
    const int r = e / nout, o = e % nout;
    if (r0 + r >= n) continue;
    const unsigned short* w = W + (size_t)o * nin;
    float acc = b[o];
    for (int i = 0; i < nin; ++i) acc = fmaf(sA[r][i], bf16_round_to_float(w[i]), acc);
    const size_t idx = (size_t)(r0 + r) * nout + o;
    if (Z) Z[idx] = acc;
    if (act) Aout[idx] = gelu(acc);
  }
}

// dA = dZ W (then times gelu'(Zprev) when act): grid ceil(n / kRows); nout <= kMaxIn.
__global__ void __launch_bounds__(256) k_linear_bwd_data(const float* __restrict__ dZ, int n, int nout,
                                                        const unsigned short* __restrict__ W, int nin,
                                                        const float* __restrict__ Zprev, int act,
                                                        float* __restrict__ dA) {
  __shared__ float sD[kRows][kMaxIn + 1];
  const int r0 = blockIdx.x * kRows;
  for (int e = threadIdx.x; e < kRows * nout; e += blockDim.x) {
    const int r = e / nout, o = e % nout;
    sD[r][o] = r0 + r < n ? dZ[(size_t)(r0 + r) * nout + o] : 0.0f;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kRows * nin; e += blockDim.x) {
    const int r = e / nin, i = e % nin;
    if (r0 + r >= n) continue;
    float acc = 0.0f;
    for (int o = 0; o < nout; ++o) acc = fmaf(sD[r][o], bf16_round_to_float(W[(size_t)o * nin + i]), acc);
    const size_t idx = (size_t)(r0 + r) * nin + i;
    dA[idx] = act ? acc * gelu_grad(Zprev[idx]) : acc;
  }
}

// Partial weight and bias gradients over chunks of kChunk samples:
//   part[c][o][i] = sum_{n in chunk} dZ[n][o] A[n][i], part[c][o][nin] = sum dZ[n][o].
// A workgroup is one job of a chunk: 64 of the wider side of the layer along its
// lanes by 16 of the other.  Half a chunk of both sides sits in LDS (40 KB, so
// that three workgroups share a CU) with the other half's loads in flight: the
// operands come from other XCDs, about a microsecond away, and a loop that loads
// 16 samples at a time spent 16 such latencies on the chunk (a backward launch of a 128 -> 128 layer at 4096
// samples: 24.8 us then, 20.1 us now; the last layer's 26.7 and 11.2 us; 26.8 us
// with whole chunks in 80 KB).  Each wave takes four of the 16; per sample one LDS read along the lanes, one broadcast and four
// FMAs.  Sums run over the samples in order (the bits of a loop over one output).
constexpr int kWu = 16;
struct BwdW {
  int L, U, lw, nu;  // wider and other side, lane groups, groups of kWu
  bool in;           // the lanes run along the inputs
};
__host__ __device__ inline BwdW bwd_w_shape(int nin, int nout) {
  BwdW b;
  b.in = nin >= nout;
  b.L = b.in ? nin : nout;
  b.U = b.in ? nout : nin;
  b.lw = (b.L + 63) / 64;
  b.nu = (b.U + kWu - 1) / kWu;
  return b;
}
constexpr int kWs = 128;  // samples of a chunk in LDS at a time
constexpr size_t kBwdWLds = sizeof(float) * kWs * (64 + kWu);

// kWs rows of src[.][ld] from row s0 on (zero from ns on), columns c0 .. c0 + W
// (zero past ld): into registers, then to dst[kWs][W].  al: 16-byte loads.
template <int W>
struct StageCols {
  float4 v[kWs * W / 1024];
  __device__ __forceinline__ void load(const float* __restrict__ src, int ld, int c0, int s0, int ns,
                                       bool al) {
#pragma unroll
    for (int k = 0; k < kWs * W / 1024; ++k) {
      const int e = (int)threadIdx.x + 256 * k, s = e / (W / 4), c = c0 + 4 * (e % (W / 4));
      const float* p = src + (size_t)(s0 + s) * ld + c;
      v[k] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (s < ns && c < ld) {
        if (al) {
          v[k] = *(const float4*)p;
        } else {
          v[k].x = p[0];
          if (c + 1 < ld) v[k].y = p[1];
          if (c + 2 < ld) v[k].z = p[2];
          if (c + 3 < ld) v[k].w = p[3];
        }
      }
    }
  }
  __device__ __forceinline__ void store(float* dst) const {
#pragma unroll
    for (int k = 0; k < kWs * W / 1024; ++k) ((float4*)dst)[threadIdx.x + 256 * k] = v[k];
  }
};

__device__ __forceinline__ void bwd_w_job(const float* __restrict__ dZ, const float* __restrict__ A,
                                          int n, int nin, int nout, int job, float* lds,
                                          float* __restrict__ part) {
  const BwdW b = bwd_w_shape(nin, nout);
  const int per = b.lw * b.nu, c = job / per, k = job % per;
  const int l0 = (k % b.lw) * 64, u0 = (k / b.lw) * kWu;
  const int s0 = c * kChunk, ns = min(n - s0, kChunk);
  float* sl = lds;              // [kWs][64]
  float* su = lds + kWs * 64;   // [kWs][kWu]
  const float* L = b.in ? A : dZ;
  const float* U = b.in ? dZ : A;
  const bool all = b.L % 4 == 0 && ((uintptr_t)L % 16) == 0;
  const bool alu = b.U % 4 == 0 && ((uintptr_t)U % 16) == 0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l = l0 + lane, uw = u0 + 4 * wave;
  // the biases beside the first lane group (lanes along the inputs), or by the
  // last wave along the lanes
  const bool bu = b.in && l0 == 0, bl = !b.in && u0 == 0 && wave == 3;
  float acc[4] = {0.f, 0.f, 0.f, 0.f}, bias[4] = {0.f, 0.f, 0.f, 0.f};
  StageCols<64> vl;
  StageCols<kWu> vu;
  vl.load(L, b.L, l0, s0, ns, all);
  vu.load(U, b.U, u0, s0, ns, alu);
  for (int h = 0; h < ns; h += kWs) {
    const int m = min(kWs, ns - h);
    __syncthreads();
    vl.store(sl);
    vu.store(su);
    __syncthreads();
    if (h + kWs < ns) {  // the rest of the chunk in flight meanwhile
      vl.load(L, b.L, l0, s0 + h + kWs, ns - h - kWs, all);
      vu.load(U, b.U, u0, s0 + h + kWs, ns - h - kWs, alu);
    }
    if (uw < b.U) {
      if (bu) {
#pragma unroll 8
        for (int s = 0; s < m; ++s) {
          const float lv = sl[s * 64 + lane];
          const float4 uv = *(const float4*)(su + s * kWu + 4 * wave);
          acc[0] = fmaf(uv.x, lv, acc[0]);
          acc[1] = fmaf(uv.y, lv, acc[1]);
          acc[2] = fmaf(uv.z, lv, acc[2]);
          acc[3] = fmaf(uv.w, lv, acc[3]);
          bias[0] += uv.x;
          bias[1] += uv.y;
          bias[2] += uv.z;
          bias[3] += uv.w;
        }
      } else {
#pragma unroll 8
        for (int s = 0; s < m; ++s) {
          const float lv = sl[s * 64 + lane];
          const float4 uv = *(const float4*)(su + s * kWu + 4 * wave);
          acc[0] = fmaf(uv.x, lv, acc[0]);
          acc[1] = fmaf(uv.y, lv, acc[1]);
          acc[2] = fmaf(uv.z, lv, acc[2]);
          acc[3] = fmaf(uv.w, lv, acc[3]);
        }
      }
    }
    if (bl) {
#pragma unroll 8
      for (int s = 0; s < m; ++s) bias[0] += sl[s * 64 + lane];
    }
  }
  float* out = part + (size_t)c * nout * (nin + 1);
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int u = uw + g;
    if (u >= b.U) break;
    if (l < b.L) out[b.in ? (size_t)u * (nin + 1) + l : (size_t)l * (nin + 1) + u] = acc[g];
    if (bu && lane == g) out[(size_t)u * (nin + 1) + nin] = bias[g];
  }
  if (bl && l < nout) out[(size_t)l * (nin + 1) + nin] = bias[0];
}

// grid: njobs.
__global__ void __launch_bounds__(256) k_bwd_w(const float* __restrict__ dZ, const float* __restrict__ A,
                                               int n, int nin, int nout, float* __restrict__ part) {
  extern __shared__ float4 mlp_lds[];
  bwd_w_job(dZ, A, n, nin, nout, blockIdx.x, (float*)mlp_lds, part);
}

// The backward step of one layer in one launch: blocks [0, nw) are the weight
// gradient's jobs (the longer ones), the others form dA = dZ W (times
// gelu'(Zprev)) as k_rows_fwd does (lane = input i, W[o][i] as pairs over o,
// K = nout); both need dZ alone.  dZ is readable up to a multiple of kRowsS past n.
template <int K, int S>
__global__ void __launch_bounds__(256) k_bwd(const float* __restrict__ dZ, const float* __restrict__ A,
                                             const unsigned short* __restrict__ W,
                                             const float* __restrict__ Zprev, int n, int nin, int nw,
                                             float* __restrict__ dA, float* __restrict__ part) {
  extern __shared__ float4 mlp_lds[];
  if ((int)blockIdx.x < nw) {
    bwd_w_job(dZ, A, n, nin, K, (int)blockIdx.x, (float*)mlp_lds, part);
    return;
  }
  const int block = (int)blockIdx.x - nw, ndata = (int)gridDim.x - nw;
  unsigned(*sw)[kMaxIn + 1] = (unsigned(*)[kMaxIn + 1]) mlp_lds;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int cw = (nin + 63) / 64;
  int r0 = (block * (4 / cw) + wave / cw) * S;
  if (r0 < n) rows_touch<K, S>(dZ + (size_t)r0 * K, lane);
  for (int i = lane; i < nin; i += 64)
#pragma unroll
    for (int k = 0; k < (K + 7) / 8; ++k) {
      const int o2 = wave + 4 * k;
      if (o2 < K / 2)
        sw[o2][i] = (unsigned)W[(size_t)2 * o2 * nin + i] | ((unsigned)W[(size_t)(2 * o2 + 1) * nin + i] << 16);
    }
  __syncthreads();
  const int c = (wave % cw) * 64 + lane, cl = c < nin ? c : nin - 1;
  const int step = ndata * (4 / cw) * S;
  for (; r0 < n; r0 += step) {
    if (r0 + step < n) rows_touch<K, S>(dZ + (size_t)(r0 + step) * K, lane);
    float z[S], acc[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      z[s] = Zprev[(size_t)(r0 + s < n ? r0 + s : r0) * nin + cl];
      acc[s] = 0.0f;
    }
    rows_loop<K, S>(dZ + (size_t)r0 * K, sw, cl, acc);
    if (c < nin) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        if (r0 + s >= n) break;
        dA[(size_t)(r0 + s) * nin + c] = acc[s] * gelu_grad(z[s]);
      }
    }
  }
}

// Per parameter of the layers in t: the gradient from the partials (in chunk
// order) when part is set, an Adam step (bias-corrected: lr_t = lr / (1 - b1^t),
// c2 = 1 / (1 - b2^t)) with the new BF16 copy when m1 is set.
struct MlpLayers {
  int n;
  int nin[8], nout[8];
  size_t off[8], part[8];  // W_l in the parameters (b_l follows it), its partials
};
__global__ void __launch_bounds__(256) k_finish(MlpLayers t, const float* __restrict__ part, int nchunks,
                                                float* __restrict__ g, float* __restrict__ p,
                                                unsigned short* __restrict__ pb, float* __restrict__ m1,
                                                float* __restrict__ m2, float lr_t, float b1, float b2,
                                                float c2, float eps) {
  size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  int l = 0;
  for (; l < t.n; ++l) {
    const size_t m = (size_t)t.nout[l] * (t.nin[l] + 1);
    if (e < m) break;
    e -= m;
  }
  if (l == t.n) return;
  const int nin = t.nin[l], nout = t.nout[l];
  const size_t per = (size_t)nout * (nin + 1), nw = (size_t)nout * nin;
  const size_t idx = t.off[l] + e;
  float gi;
  if (part) {
    // partial of W[o][i] at o (nin + 1) + i, of b[o] at o (nin + 1) + nin
    const size_t at = e < nw ? e / nin * (nin + 1) + e % nin : (e - nw) * (nin + 1) + nin;
    const float* src = part + t.part[l] + at;
    float acc = 0.0f;
#pragma unroll 16
    for (int c = 0; c < nchunks; ++c) acc += src[(size_t)c * per];
    g[idx] = gi = acc;
  } else {
    gi = g[idx];
  }
  if (m1) {
    const float a = b1 * m1[idx] + (1.0f - b1) * gi;
    const float v = b2 * m2[idx] + (1.0f - b2) * gi * gi;
    m1[idx] = a;
    m2[idx] = v;
    const float pn = p[idx] - lr_t * a / (sqrtf(v * c2) + eps);
    p[idx] = pn;
    pb[idx] = __builtin_bit_cast(unsigned short, (__bf16)pn);
  }
}

// Mean-squared error: dY = 2 (Y - T) / (n * nout); loss partial sums per block.
__global__ void __launch_bounds__(256) k_mse(const float* __restrict__ Y, const float* __restrict__ T, size_t m,
                                            float scale, float* __restrict__ dY, double* __restrict__ lossp) {
  __shared__ double red[256];
  double s = 0.0;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < m; i += (size_t)gridDim.x * blockDim.x) {
    const float d = Y[i] - T[i];
    dY[i] = 2.0f * d * scale;
    s += (double)d * d;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) lossp[blockIdx.x] = red[0];
}

// Gathers a minibatch: xb[j] = x[idx[j]], tb[j] = t[idx[j]], a thread per value.
// idx may be pinned host memory (each entry is then read over the bus).
__global__ void __launch_bounds__(256) k_gather_rows(const float* __restrict__ x,
                                                     const float* __restrict__ t,
                                                     const int* __restrict__ idx, int nb, int nin,
                                                     int nout, float* __restrict__ xb,
                                                     float* __restrict__ tb) {
  const int w = nin + nout;
  const long long e = blockIdx.x * 256LL + threadIdx.x;
  const int j = (int)(e / w), i = (int)(e % w);
  if (j >= nb) return;
  const size_t r = (size_t)idx[j];
  if (i < nin) xb[(size_t)j * nin + i] = x[r * nin + i];
  else tb[(size_t)j * nout + i - nin] = t[r * nout + i - nin];
}

int mlp_max_width() { return kMaxIn; }
int mlp_chunk() { return kChunk; }
int mlp_row_slack() { return kRowsS; }

void launch_to_bf16(const float* src, size_t n, unsigned short* dst, hipStream_t s) {
  const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(k_to_bf16, dim3(blocks), dim3(256), 0, s, src, n, dst);
  RP_HIP(hipGetLastError());
}

void launch_linear_fwd(const float* A, int n, int nin, const unsigned short* W, const float* b, int nout,
                       int act, float* Z, float* Aout, hipStream_t s) {
  RP_CHECK(nin <= kMaxIn && nout <= kMaxIn && n > 0, "MLP layer wider than 128 or empty batch");
  // the specialised kernels read W rows and (narrow outputs) inputs 16 bytes at a
  // time; with layer widths that leave either off a 16-byte boundary the general
  // kernel runs
  const bool al = ((uintptr_t)W % 16) == 0 && ((uintptr_t)A % 16) == 0;
  const bool wide = nout >= 16 && al;
  const bool big = n >= kRowsBig;
  const int per = (big ? kRowsS : kRowsS / 2) * (nout > 64 ? 2 : 4);  // samples of a workgroup and pass
  const dim3 grid(std::min((n + per - 1) / per, 2048));
#define RP_ROWS(KK)                                                                              \
  hipLaunchKernelGGL((big ? k_rows_fwd<KK, kRowsS> : k_rows_fwd<KK, kRowsS / 2>), grid, dim3(256), 0, s, A, \
                     n, W, b, nout, Z, act ? Aout : nullptr)
  if (wide && nin == 128) RP_ROWS(128);
  else if (wide && nin == 64) RP_ROWS(64);
  else if (wide && nin == 32) RP_ROWS(32);
  else if (wide && nin == 16) RP_ROWS(16);
  else if (wide && nin == 8) RP_ROWS(8);
  else if (nout < 16 && nin % 4 == 0 && al)
    hipLaunchKernelGGL(k_narrow_fwd, dim3((n + 63) / 64), dim3(64), 0, s, A, n, nin, W, b, nout, act, Z,
                       Aout, (const float*)nullptr, 0.0f, (float*)nullptr, (double*)nullptr);
  else
    hipLaunchKernelGGL(k_linear_fwd, dim3((n + kRows - 1) / kRows), dim3(256), 0, s, A, n, nin, W, b, nout,
                       act, Z, Aout);
#undef RP_ROWS
  RP_HIP(hipGetLastError());
}

// The output layer with the mean-squared error: Y, dY and the loss partials
// (nlossp of them at most: launch_output_loss_blocks).
int launch_output_loss_blocks(int n, int nout) {
  return nout < 16 ? (n + 63) / 64 : (int)std::min<size_t>(((size_t)n * nout + 255) / 256, 1024);
}
void launch_output_loss(const float* A, int n, int nin, const unsigned short* W, const float* b, int nout,
                        const float* T, float scale, float* Y, float* dY, double* lossp, hipStream_t s) {
  const int nlossp = launch_output_loss_blocks(n, nout);
  const bool al = ((uintptr_t)W % 16) == 0 && ((uintptr_t)A % 16) == 0;
  if (nout < 16 && nin % 4 == 0 && al) {
    hipLaunchKernelGGL(k_narrow_fwd, dim3(nlossp), dim3(64), 0, s, A, n, nin, W, b, nout, 0, Y,
                       (float*)nullptr, T, scale, dY, lossp);
  } else {
    launch_linear_fwd(A, n, nin, W, b, nout, 0, Y, nullptr, s);
    hipLaunchKernelGGL(k_mse, dim3(nlossp), dim3(256), 0, s, Y, T, (size_t)n * nout, scale, dY, lossp);
  }
  RP_HIP(hipGetLastError());
}

// Backward step of one layer: the weight-gradient partials, and with dA also
// dA = dZ W gelu'(Zprev).
void launch_bwd_layer(const float* dZ, const float* A, int n, int nin, int nout, const unsigned short* W,
                      const float* Zprev, float* dA, float* part, hipStream_t s) {
  RP_CHECK(nin <= kMaxIn && nout <= kMaxIn && n > 0, "MLP layer wider than 128 or empty batch");
  const BwdW b = bwd_w_shape(nin, nout);
  const int nw = (n + kChunk - 1) / kChunk * b.lw * b.nu;  // weight-gradient jobs
  const bool big = n >= kRowsBig;
  const int per = (big ? kRowsS : kRowsS / 2) * (nin > 64 ? 2 : 4);
  const int nd = std::min((n + per - 1) / per, 2048);
  auto weights = [&] {
    RP_HIP(hipFuncSetAttribute((const void*)k_bwd_w, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)kBwdWLds));
    hipLaunchKernelGGL(k_bwd_w, dim3(nw), dim3(256), kBwdWLds, s, dZ, A, n, nin, nout, part);
  };
  auto both = [&](auto kernel) {
    RP_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)kBwdWLds));
    hipLaunchKernelGGL(kernel, dim3(nd + nw), dim3(256), kBwdWLds, s, dZ, A, W, Zprev, n, nin, nw, dA, part);
  };
  // a kernel of its own for the widths of hidden layers and the closure's two outputs;
  // any other width (an output layer of a network that is not the closure's) runs the
  // two general kernels
#define RP_BWD(KK) \
  case KK: both(big ? k_bwd<KK, kRowsS> : k_bwd<KK, kRowsS / 2>); break;
  if (!dA) {
    weights();
  } else {
    switch (nout) {
      RP_BWD(2) RP_BWD(8) RP_BWD(16) RP_BWD(32) RP_BWD(64) RP_BWD(128)
      default:
        weights();
        hipLaunchKernelGGL(k_linear_bwd_data, dim3((n + kRows - 1) / kRows), dim3(256), 0, s, dZ, n, nout,
                           W, nin, Zprev, 1, dA);
    }
  }
#undef RP_BWD
  RP_HIP(hipGetLastError());
}

// Layers [l0, l1) (dims[l0 ..], W_l at woff[l]): gradients from part (unless
// null; layer l's partials at poff[l - l0]) and, with m1, an Adam step.
void launch_finish(int l0, int l1, const int* dims, const size_t* woff, const size_t* poff,
                   const float* part, int nchunks, float* g, float* p, unsigned short* pb, float* m1,
                   float* m2, float lr_t, float b1, float b2, float c2, float eps, hipStream_t s) {
  for (int a = l0; a < l1; a += 8) {
    MlpLayers t;
    t.n = std::min(8, l1 - a);
    size_t tot = 0;
    for (int i = 0; i < t.n; ++i) {
      t.nin[i] = dims[a + i];
      t.nout[i] = dims[a + i + 1];
      t.off[i] = woff[a + i];
      t.part[i] = part ? poff[a + i - l0] : 0;
      tot += (size_t)t.nout[i] * (t.nin[i] + 1);
    }
    hipLaunchKernelGGL(k_finish, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, t, part, nchunks, g,
                       p, pb, m1, m2, lr_t, b1, b2, c2, eps);
  }
  RP_HIP(hipGetLastError());
}

void launch_gather_rows(const float* x, const float* t, const int* idx, int nb, int nin, int nout, float* xb,
                        float* tb, hipStream_t s) {
  const long long m = (long long)nb * (nin + nout);
  hipLaunchKernelGGL(k_gather_rows, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, s, x, t, idx, nb, nin, nout, xb, tb);
  RP_HIP(hipGetLastError());
}

}  // namespace rp
