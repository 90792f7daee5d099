// Shift predictor: a small tanh MLP trained and evaluated on the GPU.
//
// Network: nin inputs -> `depth` hidden layers of `width` tanh units -> nout
// linear outputs.  Master weights, inputs and outputs are FP32; every matrix
// product runs on the matrix cores with BF16 operands (round to nearest even)
// and FP32 accumulation (v_mfma_f32_16x16x16bf16_1k).  Inputs are mapped
// x' = (x - in_shift) * in_scale and outputs y = y' / out_scale + out_shift,
// so training sees O(1) numbers.
//
// A pass is one launch: a work-group carries 16 rows through every layer
// (k_mlp_rows), and a training step adds one launch for the sums over rows
// with the Adam update in its epilogue (k_mlp_grad).  The networks are small
// (37k to 140k weights), so a step is bound by launches and by the latency of
// its dependent phases, not by arithmetic: per-layer GEMM launches with their
// own gather, bias-sum, loss and Adam launches took 649 us a step at batch
// 1024 and width 128 (of which 490 us the bias sums, one thread walking the
// batch), these two 28 us.  A prediction of 8191 rows at width 256 went from
// 411 to 42 us, of 12 rows from 72 to 24 us (pinned host rows read and
// written in place, one launch, one wait).
//
// Flat parameter layout (FP32), dimensions padded to multiples of 16
// (nin_p = pad16(nin), nout_p = pad16(nout); padded rows/columns stay zero):
//   W_0 [width x nin_p], b_0 [width],
//   W_l [width x width], b_l [width]            l = 1 .. depth-1
//   W_o [nout_p x width], b_o [nout_p]
// W is row-major by output unit: W[o * in + i].
#include "common.h"
#include <algorithm>

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline short to_bf16(float x) {
  unsigned u = __float_as_uint(x);
  u += 0x7fffu + ((u >> 16) & 1u);        // round to nearest even (finite inputs)
  return (short)(u >> 16);
}

#define MLP_T 1024       // most threads of a 16-row tile (mlp_threads)
#define MLP_WMAX 512     // widest layer
#define MLP_LMAX 9       // 8 hidden layers and the output layer
#define MLP_KU 8         // depth-16 steps whose operands are loaded together

// Offsets of one network (floats of the flat parameters) and its sizes.
struct MlpNet {
  int nin, nin_p, width, depth, nout, nout_p;
  int off_w[MLP_LMAX], off_b[MLP_LMAX];
};

// Threads of k_mlp_rows: a wave per 16-column tile of a layer, eight to sixteen.
// A batch of few rows runs on few CUs, each reading every weight (1 MB a layer
// at width 512) through its own memory path, so bytes in flight per CU are
// what counts.  64 inputs, width 512, eight layers: 16 rows took 244 us with
// eight waves and the weights by operand order, where one launch per layer
// over all CUs had taken 181; 187 with the loads along rows, 119 with sixteen
// waves too (a step of 16 rows 402, 308, 344, 248).  Width 256, three layers:
// 36, 80, 29, 26.
inline int mlp_threads(const MlpNet &N) { return std::min(MLP_T, std::max(512, 4 * N.width)); }

__device__ inline unsigned mlp_hash(unsigned long long seed, unsigned a, unsigned b) {
  unsigned long long h = seed ^ (0x9E3779B97F4A7C15ull * (a + 1)) ^ (0xC2B2AE3D27D4EB4Full * (b + 7));
  h ^= h >> 33; h *= 0xff51afd7ed558ccdull; h ^= h >> 33; h *= 0xc4ceb9fe1a85ec53ull; h ^= h >> 33;
  return (unsigned)h;
}

// One 16 x 16 tile of A W: A the 16 rows of bf16 activations in LDS, K long
// (a multiple of 16); W(k, n) = w[n ldn + k] (TRANS false: the forward
// product, four consecutive weights per lane) or w[k ldn + n] (TRANS true: the
// product with the transposed layer of the backward pass).  Lane l supplies
// A[l % 16][k0 + 4 (l / 16) + j] and W(k0 + 4 (l / 16) + j, n0 + l % 16), j < 4;
// accumulator register i is entry (4 (l / 16) + i, l % 16).  The weights of
// MLP_KU steps are loaded before the first is used, from clamped in-range
// steps, so a pass costs one memory latency per 128 of K.  In the forward
// product four consecutive lanes load 64 consecutive bytes of a weight row
// (lane l row l / 4) and the BF16 values change lanes afterwards; with the
// rows on consecutive lanes, as the operand has them, a load of the wave met
// sixteen rows and a CU took in some 15 bytes a cycle.
template <bool TRANS>
__device__ inline f32x4 mlp_tile(const short (*__restrict__ A)[MLP_WMAX + 8], int K, const float *__restrict__ w, int ldn,
                                 int n0) {
  const int l = threadIdx.x & 63, r = l & 15, q = 4 * (l >> 4);
  const int from = 4 * (4 * r + (l >> 4));           // byte index of the lane that loaded this lane's weights
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int kb = 0; kb < K; kb += 16 * MLP_KU) {
    f32x4 wv[MLP_KU];
#pragma unroll
    for (int s = 0; s < MLP_KU; ++s) {
      const int k = min(kb + 16 * s, K - 16);
      if (TRANS) {
#pragma unroll
        for (int j = 0; j < 4; ++j) wv[s][j] = w[(size_t)(k + q + j) * ldn + n0 + r];
      } else {
        wv[s] = *(const f32x4 *)(w + (size_t)(n0 + (l >> 2)) * ldn + k + 4 * (l & 3));
      }
    }
#pragma unroll
    for (int s = 0; s < MLP_KU; ++s) {
      const int k = kb + 16 * s;
      if (k < K) {
        const bf16x4 a = *(const bf16x4 *)&A[r][k + q];
        bf16x4 b;
#pragma unroll
        for (int j = 0; j < 4; ++j) b[j] = to_bf16(wv[s][j]);
        if (!TRANS) {
          union { bf16x4 h; int d[2]; } u;
          u.h = b;
          u.d[0] = __builtin_amdgcn_ds_bpermute(from, u.d[0]);
          u.d[1] = __builtin_amdgcn_ds_bpermute(from, u.d[1]);
          b = u.h;
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
      }
    }
  }
  return acc;
}

// Rows b0 .. b0 + 15 (b0 = 16 blockIdx.x) through the whole network, the
// activations of the tile in LDS as the bf16 operands of the next layer.
//
// TRAIN false (prediction): x holds raw rows (n x nin) and y receives the
// scaled outputs (n x nout); rows past n are zeros and are not stored.
//
// TRAIN true: row b is row idx(b) of the normalised set (X: n x nin_p, T: n x
// nout), idx(b) = b when B == n (the whole set, in order), else a hashed draw
// with replacement from (seed, step, b).  After the forward pass come the
// mean squared error over the nout real outputs, its gradient dY = 2 (Y - T) /
// (B nout) and the backward pass to dZ of every hidden layer.  For the sums
// over rows (k_mlp_grad) it leaves the bf16 operands transposed, [column][B],
// which are the four consecutive rows each lane holds (one 8-byte store):
// actT (input, then the hidden layers) and dzT (hidden layers, then dY); the
// column sums of dZ and dY over its rows in part[tile][column] (FP32 values,
// columns as dzT) and the tile's squared error in losspart.  act32 keeps the
// FP32 activations for tanh' in the order the same lane reads them back.
template <bool TRAIN>
__global__ __launch_bounds__(MLP_T) void k_mlp_rows(MlpNet N, const float *__restrict__ p, const float *__restrict__ scl,
                                                    const float *__restrict__ x, float *__restrict__ y, int n, int B,
                                                    const float *__restrict__ T, unsigned long long seed, int step,
                                                    short *__restrict__ actT, short *__restrict__ dzT,
                                                    float *__restrict__ act32, float *__restrict__ part,
                                                    float *__restrict__ losspart) {
  __shared__ __align__(16) short s_a[2][16][MLP_WMAX + 8];   // 8 shorts of padding: rows start on different banks
  __shared__ int s_src[16];
  const int NT = blockDim.x, NW = NT / 64;
  const int t = threadIdx.x, w = t >> 6, l = t & 63, r = l & 15, q = 4 * (l >> 4);
  const int b0 = blockIdx.x * 16, W = N.width, L = N.depth;
  if (TRAIN) {
    if (t < 16) s_src[t] = (B == n) ? b0 + t : (int)(mlp_hash(seed, (unsigned)step, (unsigned)(b0 + t)) % (unsigned)n);
    __syncthreads();
  }
  for (int e = t; e < 16 * N.nin_p; e += NT) {
    const int row = e / N.nin_p, i = e - row * N.nin_p;
    float v = 0.f;
    if (TRAIN) v = x[(size_t)s_src[row] * N.nin_p + i];
    else if (i < N.nin) v = ((b0 + row < n ? x[(size_t)(b0 + row) * N.nin + i] : 0.f) - scl[i]) * scl[N.nin_p + i];
    s_a[0][row][i] = to_bf16(v);
    if (TRAIN) actT[(size_t)i * B + b0 + row] = to_bf16(v);
  }
  __syncthreads();
  int cur = 0;
  for (int lay = 0; lay < L; ++lay) {
    const int in = lay ? W : N.nin_p;
    for (int n0 = 16 * w; n0 < W; n0 += 16 * NW) {
      const float bias = p[N.off_b[lay] + n0 + r];
      f32x4 v = mlp_tile<false>(s_a[cur], in, p + N.off_w[lay], in, n0);
      bf16x4 h;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] = tanhf(v[i] + bias);
        h[i] = to_bf16(v[i]);
        s_a[1 - cur][q + i][n0 + r] = h[i];
      }
      if (TRAIN) {
        *(bf16x4 *)(actT + (size_t)(N.nin_p + lay * W + n0 + r) * B + b0 + q) = h;
        *(f32x4 *)(act32 + ((size_t)lay * B + b0) * W + n0 * 16 + 4 * l) = v;
      }
    }
    cur = 1 - cur;
    __syncthreads();
  }
  // output layer: one tile (nout_p = 16), wave 0
  if (w == 0) {
    const float bias = p[N.off_b[L] + r];
    f32x4 v = mlp_tile<false>(s_a[cur], W, p + N.off_w[L], W, 0);
    if (!TRAIN) {
      const float *out_shift = scl + 2 * N.nin_p, *out_scale = out_shift + 16;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (r < N.nout && b0 + q + i < n) y[(size_t)(b0 + q + i) * N.nout + r] = (v[i] + bias) / out_scale[r] + out_shift[r];
    } else {
      const float sc = 2.f / (float)(B * N.nout);
      float ls = 0.f, cs = 0.f;
      bf16x4 h;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float g = 0.f;
        if (r < N.nout) {
          const float d = v[i] + bias - T[(size_t)s_src[q + i] * N.nout + r];
          ls += d * d;
          g = sc * d;
        }
        h[i] = to_bf16(g);
        s_a[1 - cur][q + i][r] = h[i];
        cs += g;
      }
      *(bf16x4 *)(dzT + (size_t)(L * W + r) * B + b0 + q) = h;
      cs += __shfl_xor(cs, 16);
      cs += __shfl_xor(cs, 32);
      if (l < 16) part[(size_t)blockIdx.x * (L * W + 16) + L * W + r] = cs;
      for (int off = 32; off > 0; off >>= 1) ls += __shfl_xor(ls, off);
      if (l == 0) losspart[blockIdx.x] = ls;
    }
  }
  if (!TRAIN) return;
  cur = 1 - cur;
  __syncthreads();
  // backward: dZ of hidden layer lay from the layer above it
  for (int lay = L - 1; lay >= 0; --lay) {
    const int K = (lay == L - 1) ? N.nout_p : W;
    for (int n0 = 16 * w; n0 < W; n0 += 16 * NW) {
      const f32x4 a = *(const f32x4 *)(act32 + ((size_t)lay * B + b0) * W + n0 * 16 + 4 * l);
      f32x4 v = mlp_tile<true>(s_a[cur], K, p + N.off_w[lay + 1], W, n0);
      bf16x4 h;
      float cs = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] *= 1.f - a[i] * a[i];
        h[i] = to_bf16(v[i]);
        s_a[1 - cur][q + i][n0 + r] = h[i];
        cs += v[i];
      }
      *(bf16x4 *)(dzT + (size_t)(lay * W + n0 + r) * B + b0 + q) = h;
      cs += __shfl_xor(cs, 16);
      cs += __shfl_xor(cs, 32);
      if (l < 16) part[(size_t)blockIdx.x * (L * W + 16) + lay * W + n0 + r] = cs;
    }
    cur = 1 - cur;
    __syncthreads();
  }
}

// Adam (Kingma & Ba 2015) on one parameter, step t >= 1.
__device__ inline void mlp_adam(float gi, float *__restrict__ p, float *__restrict__ m, float *__restrict__ v, float lr,
                                float b1, float b2, float eps, int t) {
  const float mi = b1 * *m + (1.f - b1) * gi;
  const float vi = b2 * *v + (1.f - b2) * gi * gi;
  *m = mi;
  *v = vi;
  const float mh = mi / (1.f - powf(b1, (float)t)), vh = vi / (1.f - powf(b2, (float)t));
  *p -= lr * mh / (sqrtf(vh) + eps);
}

// The gradient over the B rows of a batch from what k_mlp_rows<true> left,
// one wave per 16 x 16 tile of a weight matrix: dW(o, i) = sum_b dZ(b, o)
// act(b, i), the K = B chain of one accumulator in row order (64 matrix
// instructions at B = 1024, 0.5 us; splitting it would only reorder the sum),
// its operands loaded MLP_GU depth-16 steps ahead.  tiles[4 k ..]: first dzT
// row, first actT row, parameter offset of entry (0, 0), row stride.  The
// blocks after the tiles take the biases (one thread per column of part, the
// tiles' sums in row order) and the last one the loss.  grad != nullptr
// stores the gradient; else the parameter is updated (Adam, step t).
#define MLP_GU 16
__global__ __launch_bounds__(64) void k_mlp_grad(MlpNet N, int B, int ntile, const int *__restrict__ tiles,
                                                 const short *__restrict__ dzT, const short *__restrict__ actT,
                                                 const float *__restrict__ part, const float *__restrict__ losspart,
                                                 float *__restrict__ grad, float *__restrict__ p, float *__restrict__ m,
                                                 float *__restrict__ v, float lr, int t, float *__restrict__ loss,
                                                 int hist_slot) {
  const int l = threadIdx.x, ncol = N.depth * N.width + 16, nb = B / 16;
  const int blk = blockIdx.x;
  auto finish = [&](int e, float g) {
    if (grad) grad[e] = g;
    else mlp_adam(g, p + e, m + e, v + e, lr, 0.9f, 0.999f, 1e-8f, t);
  };
  if (blk < ntile) {
    const int r = l & 15, q = 4 * (l >> 4);
    const short *a = dzT + (size_t)(tiles[4 * blk] + r) * B + q, *b = actT + (size_t)(tiles[4 * blk + 1] + r) * B + q;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int kb = 0; kb < B; kb += 16 * MLP_GU) {
      bf16x4 av[MLP_GU], bv[MLP_GU];
#pragma unroll
      for (int s = 0; s < MLP_GU; ++s) {
        const int k = min(kb + 16 * s, B - 16);
        av[s] = *(const bf16x4 *)(a + k);
        bv[s] = *(const bf16x4 *)(b + k);
      }
#pragma unroll
      for (int s = 0; s < MLP_GU; ++s)
        if (kb + 16 * s < B) acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av[s], bv[s], acc, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) finish(tiles[4 * blk + 2] + (q + i) * tiles[4 * blk + 3] + r, acc[i]);
    return;
  }
  const int col = (blk - ntile) * 64 + l;
  if (col < ncol) {
    float s = 0.f;
#pragma unroll 16
    for (int k = 0; k < nb; ++k) s += part[(size_t)k * ncol + col];
    const int lay = col / N.width < N.depth ? col / N.width : N.depth;
    finish(N.off_b[lay] + col - lay * N.width, s);
  }
  if (blk == ntile) {
    float s = 0.f;
    for (int k = l; k < nb; k += 64) s += losspart[k];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (l == 0) {
      s /= (float)(B * N.nout);
      loss[0] = s;
      if (hist_slot >= 0) loss[1 + hist_slot] = s;
    }
  }
}

// x' = (x - shift) * scale into rows of nin_p (zeros beyond nin); likewise
// for targets when T != nullptr.  grid: rows.
__global__ __launch_bounds__(64) void k_mlp_normalize(int nin, int nin_p, int nout, const float *__restrict__ x,
                                                      const float *__restrict__ t, const float *__restrict__ scl,
                                                      float *__restrict__ xo, float *__restrict__ to) {
  const int b = blockIdx.x, i = threadIdx.x;
  const float *in_shift = scl, *in_scale = scl + nin_p, *out_shift = scl + 2 * nin_p;
  const float *out_scale = out_shift + 16;
  if (i < nin_p) xo[(size_t)b * nin_p + i] = (i < nin) ? (x[(size_t)b * nin + i] - in_shift[i]) * in_scale[i] : 0.f;
  if (t && i < nout) to[(size_t)b * nout + i] = (t[(size_t)b * nout + i] - out_shift[i]) * out_scale[i];
}

// Glorot-uniform weights from a hash of (seed, index), zero biases and zero
// padding.  One thread per parameter.
__global__ __launch_bounds__(256) void k_mlp_init(int np, float *__restrict__ p, const int *__restrict__ meta,
                                                  int nseg, unsigned long long seed) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= np) return;
  // meta: per segment {offset, rows, cols, real_rows, real_cols, is_bias}
  float v = 0.f;
  for (int s = 0; s < nseg; ++s) {
    const int *d = meta + 6 * s;
    const int off = d[0], rows = d[1], cols = d[2];
    if (i < off || i >= off + rows * cols) continue;
    const int e = i - off, rr = e / cols, cc = e - rr * cols;
    if (!d[5] && rr < d[3] && cc < d[4]) {
      const float a = sqrtf(6.f / (float)(d[3] + d[4]));
      const float u = (float)(mlp_hash(seed, (unsigned)i, 0x51u) >> 8) * (1.f / 16777216.f);
      v = (2.f * u - 1.f) * a;
    }
  }
  p[i] = v;
}
