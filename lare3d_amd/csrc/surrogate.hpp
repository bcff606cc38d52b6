// surrogate.hpp -- learned conduction surrogate: a 3x3x3-stencil MLP that
// predicts the temperature increment of one whole RKL2 super-step
// (conduct.f90:39 conduct_heat), with BF16 MFMA inference and training
// kernels (FP32 accumulation) and a trapezoidal residual check that sends a
// step back to the plain RKL2 solver when it fails.  No reference
// counterpart.
//
// Network: x (27 neighbours x 12 channels = 324, channels 10 and 11 zero,
//   padded with zeros to K = 336 = 21 MFMA steps)
//   -> W1 (336 x 64) + b1 -> GELU -> W2 (64 x 64) + b2 -> GELU -> W3 (64) + b3
//   -> y, with dT = y * y_scale.
// Channels of a cell (standardised with the stored mean / std):
//   0 T, 1-3 unit vector of the cell-centred B, 4 rho, 5 log dt, 6 |B|,
//   7-9 centred differences of T along x, y, z.
//
// MFMA layout used throughout (v_mfma_f32_16x16x16_bf16, 64 lanes, l = lane):
//   A (16 x 16, rows m, cols k): lane l holds A[l % 16][4 (l / 16) + r], r = 0..3
//   B (16 x 16, rows k, cols n): lane l holds B[4 (l / 16) + r][l % 16]
//   D (16 x 16):                 lane l holds D[4 (l / 16) + r][l % 16]
// D has the layout of B, so a layer computed as (W^T)(H^T) feeds the next
// layer's B operand from registers, with no transpose through LDS.

#define SUR_CH 12            // channels stored per cell (10 used)
#define SUR_NCH 10
#define SUR_KREAL 324        // 27 * SUR_CH
#define SUR_K 336            // SUR_KREAL padded to a multiple of 16
#define SUR_H 64
#define SUR_KP 344           // padded LDS row of W1^T (bf16 elements)
#define SUR_HP 72            // padded LDS row of W2^T
// parameter vector (float): W1[k][f], b1[f], W2[k][f], b2[f], W3[f], b3
#define SUR_OFF_W1 0
#define SUR_OFF_B1 (SUR_K * SUR_H)
#define SUR_OFF_W2 (SUR_OFF_B1 + SUR_H)
#define SUR_OFF_B2 (SUR_OFF_W2 + SUR_H * SUR_H)
#define SUR_OFF_W3 (SUR_OFF_B2 + SUR_H)
#define SUR_OFF_B3 (SUR_OFF_W3 + SUR_H)
#define SUR_NPARAM (SUR_OFF_B3 + 1)

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even (finite inputs).
__device__ __forceinline__ unsigned short f2bf(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ bf16x4 pack4(float a, float b, float c, float d) {
  bf16x4 v;
  v[0] = (short)f2bf(a);
  v[1] = (short)f2bf(b);
  v[2] = (short)f2bf(c);
  v[3] = (short)f2bf(d);
  return v;
}

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float x) {
  const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
  const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
  return cdf + x * pdf;
}

struct SurNorm {
  float mu[SUR_CH], sd[SUR_CH];
  float y_scale;
};

// Cell channels over cells 0..n+1 (box b).  Temperature T = tfac * e
// (conduct.f90:72-73 with xi_n = 0 and zero ionisation energy).
__global__ __launch_bounds__(BX * BY) void k_sur_features(Geo g, Box b, const real *__restrict__ energy,
                                                          const real *__restrict__ rho,
                                                          const double *__restrict__ bx,
                                                          const double *__restrict__ by,
                                                          const double *__restrict__ bz, float *__restrict__ feat,
                                                          SurNorm nm, double tfac, double logdt, int normalise) {
  BOX_INDEX(b, i, j, k);
  const int c = g.idx(i, j, k);
  const int X = 1, Y = g.sy, Z = g.sz;
  const double T = tfac * energy[c];
  const double b1x = (bx[c] + bx[c - X]) * 0.5;
  const double b1y = (by[c] + by[c - Y]) * 0.5;
  const double b1z = (bz[c] + bz[c - Z]) * 0.5;
  const double bm = sqrt(b1x * b1x + b1y * b1y + b1z * b1z);
  const double inv = 1.0 / (bm > 1.0e-30 ? bm : 1.0e-30);
  const double gx = tfac * (energy[c + X] - energy[c - X]) / (g.dxc[i] + g.dxc[i - 1]);
  const double gy = tfac * (energy[c + Y] - energy[c - Y]) / (g.dyc[j] + g.dyc[j - 1]);
  const double gz = tfac * (energy[c + Z] - energy[c - Z]) / (g.dzc[k] + g.dzc[k - 1]);
  float v[SUR_CH] = {(float)T, (float)(b1x * inv), (float)(b1y * inv), (float)(b1z * inv), (float)rho[c],
                     (float)logdt, (float)bm, (float)gx, (float)gy, (float)gz, 0.0f, 0.0f};
  float *o = feat + (size_t)c * SUR_CH;
#pragma unroll
  for (int q = 0; q < SUR_CH; ++q) o[q] = (normalise && q < SUR_NCH) ? (v[q] - nm.mu[q]) / nm.sd[q] : v[q];
}

// Neighbour q (0..26) of a stencil as a linear offset: q = 9 (dz+1) + 3 (dy+1) + (dx+1).
__device__ __forceinline__ int nb_offset(const Geo &g, int q) {
  return (q / 9 - 1) * g.sz + ((q / 3) % 3 - 1) * g.sy + (q % 3 - 1);
}

// splitmix64 hash (public-domain mixing function of Steele, Lea and Flood).
__host__ __device__ __forceinline__ unsigned long long mix64(unsigned long long x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

// Interior cells for rows [0, rows) of a sample (cells[r] = linear index),
// drawn by hash of (seed, r).  Even rows are uniform; odd rows take the
// most active of 8 uniform candidates, scored by the discrete Laplacian
// |6 T - sum of the 6 face neighbours| of the raw temperature channel, so
// that the cells where conduction acts are well represented.
__device__ __forceinline__ int sample_cell(const Geo &g, unsigned long long h) {
  const int i = 1 + (int)((h & 0xFFFFFull) % (unsigned long long)g.nx);
  const int j = 1 + (int)(((h >> 20) & 0xFFFFFull) % (unsigned long long)g.ny);
  const int k = 1 + (int)(((h >> 40) & 0xFFFFFull) % (unsigned long long)g.nz);
  return g.idx(i, j, k);
}
__global__ void k_sur_sample_cells(Geo g, const float *__restrict__ feat, unsigned long long seed, int rows,
                                   int *__restrict__ cells) {
  const int r = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (r >= rows) return;
  const unsigned long long h = mix64(seed * 0x100000001B3ull + (unsigned long long)r);
  int best = sample_cell(g, h);
  if (r & 1) {
    float score = -1.0f;
    for (int t = 0; t < 8; ++t) {
      const int c = sample_cell(g, mix64(h + (unsigned long long)(t + 1)));
      const float T = feat[(size_t)c * SUR_CH];
      const float lap = 6.0f * T - feat[(size_t)(c + 1) * SUR_CH] - feat[(size_t)(c - 1) * SUR_CH] -
                        feat[(size_t)(c + g.sy) * SUR_CH] - feat[(size_t)(c - g.sy) * SUR_CH] -
                        feat[(size_t)(c + g.sz) * SUR_CH] - feat[(size_t)(c - g.sz) * SUR_CH];
      const float sc = fabsf(lap);
      if (sc > score) {
        score = sc;
        best = c;
      }
    }
  }
  cells[r] = best;
}

// X[base + r][q * 12 + ch] = feat[cells[r] + off(q)][ch]
__global__ void k_sur_gather(Geo g, const float *__restrict__ feat, const int *__restrict__ cells, int rows,
                             float *__restrict__ Xout) {
  const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (t >= rows * SUR_K) return;
  const int r = t / SUR_K, kk = t % SUR_K;
  const int q = kk / SUR_CH, ch = kk % SUR_CH;
  Xout[t] = kk < SUR_KREAL ? feat[(size_t)(cells[r] + nb_offset(g, q)) * SUR_CH + ch] : 0.0f;
}

// target dT of the sampled cells after one plain super-step
__global__ void k_sur_target(const real *__restrict__ E0, const real *__restrict__ E1,
                             const int *__restrict__ cells, int rows, double tfac, float *__restrict__ y) {
  const int r = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (r >= rows) return;
  const int c = cells[r];
  y[r] = (float)(tfac * (E1[c] - E0[c]));
}

// standardise stored raw rows in place: x = (x - mu) / sd per channel; y /= y_scale
__global__ void k_sur_standardise(float *__restrict__ X, float *__restrict__ y, int rows, SurNorm nm) {
  const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (t < rows * SUR_K) {
    const int kk = t % SUR_K, ch = kk % SUR_CH;
    X[t] = (kk < SUR_KREAL && ch < SUR_NCH) ? (X[t] - nm.mu[ch]) / nm.sd[ch] : 0.0f;
  }
  if (t < rows) y[t] = y[t] / nm.y_scale;
}

// ----------------------------------------------------------------------------
// training
// ----------------------------------------------------------------------------
// A mini-batch takes two launches: k_sur_fb runs forward and backward through
// the network, 16 columns per block, and k_sur_grads forms every parameter
// gradient (and applies Adam).  On batches of some hundred rows it is all
// latency; the sixteen launches of separate products, activations, row sums
// and the update took 78 us per step of 512 rows, these two take 22.
//
// Products have BF16 operands (rounded from FP32) and FP32 accumulation, K in
// steps of 16 in order; everything else is FP32.

// Columns of one mini-batch and what k_sur_fb leaves for k_sur_grads,
// feature-major rows of length nb (a multiple of 16).
struct SurBatch {
  const float *X, *y;        // rows of SUR_K inputs; targets, or NULL
  int *row;                  // row of X (and y) of each column
  float *H1, *H2, *dZ1, *dZ2;
  float *yo, *dy;
  int nb, nreal;             // columns; those that are rows (the rest is padding)
};

// Forward and, with a target, backward over 16 columns.  Wave w holds features
// 16 w .. 16 w + 15: the fragment that the MFMA leaves in its registers is the
// K step w of the next product's B operand, so layers pass BF16 fragments
// through LDS.  With draw >= 0 rows are given, column b takes row
// hash(seed, b) % draw and keeps it in row[]; otherwise row b, and the
// padding columns zeros.
// All weights but layer 1's are loaded ahead of the products that need them.
// The loads of layer 1's SUR_FB_K steps are issued together.
#define SUR_FB_K (SUR_K / 16)
__global__ __launch_bounds__(256) void k_sur_fb(SurBatch s, const float *__restrict__ w, int draw,
                                                unsigned long long seed) {
  __shared__ bf16x4 frag[2][4][64];
  __shared__ float sh2[SUR_H][17], sdy[16], sw3[SUR_H];
  const int l = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
  const int col = l & 15, kq = 4 * (l >> 4);
  const int b = (int)blockIdx.x * 16 + col;
  const bool real_row = b < s.nreal;
  int r = b;
  if (draw > 0) {
    r = (int)(mix64(seed + (unsigned long long)b) % (unsigned long long)draw);
    if (threadIdx.x < 16) s.row[b] = r;
  }
  const int f0 = wave * 16;
  bf16x4 w2f[4], w2b[4];  // W2 for the forward and the backward product
  float b1[4], b2[4], w3[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    const float *pf = w + SUR_OFF_W2 + (kk * 16 + kq) * SUR_H + f0 + col;
    w2f[kk] = pack4(pf[0], pf[SUR_H], pf[2 * SUR_H], pf[3 * SUR_H]);
    const float *pb = w + SUR_OFF_W2 + (f0 + col) * SUR_H + kk * 16 + kq;
    w2b[kk] = pack4(pb[0], pb[1], pb[2], pb[3]);
    b1[kk] = w[SUR_OFF_B1 + f0 + kq + kk];
    b2[kk] = w[SUR_OFF_B2 + f0 + kq + kk];
    w3[kk] = w[SUR_OFF_W3 + f0 + kq + kk];
  }
  const float b3 = w[SUR_OFF_B3];
  if (threadIdx.x < SUR_H) sw3[threadIdx.x] = w[SUR_OFF_W3 + threadIdx.x];
  const float tgt = s.y && real_row ? s.y[r] : 0.0f;
  // layer 1
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  float wa[SUR_FB_K][4];
  float4 xb[SUR_FB_K];
#pragma unroll
  for (int q = 0; q < SUR_FB_K; ++q) {
    const int kb = q * 16 + kq;
#pragma unroll
    for (int t = 0; t < 4; ++t) wa[q][t] = w[SUR_OFF_W1 + (kb + t) * SUR_H + f0 + col];
    xb[q] = real_row ? *(const float4 *)(s.X + (size_t)r * SUR_K + kb) : float4{0.0f, 0.0f, 0.0f, 0.0f};
  }
#pragma unroll
  for (int q = 0; q < SUR_FB_K; ++q)
    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(pack4(wa[q][0], wa[q][1], wa[q][2], wa[q][3]),
                                                    pack4(xb[q].x, xb[q].y, xb[q].z, xb[q].w), acc, 0, 0, 0);
  float z1[4], h[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    z1[t] = acc[t] + b1[t];
    h[t] = gelu(z1[t]);
    if (s.y) s.H1[(size_t)(f0 + kq + t) * s.nb + b] = h[t];
  }
  frag[0][wave][l] = pack4(h[0], h[1], h[2], h[3]);
  __syncthreads();
  // layer 2
  acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)
    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w2f[kk], frag[0][kk][l], acc, 0, 0, 0);
  float z2[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    z2[t] = acc[t] + b2[t];
    h[t] = gelu(z2[t]);
    sh2[f0 + kq + t][col] = h[t];
    if (s.y) s.H2[(size_t)(f0 + kq + t) * s.nb + b] = h[t];
  }
  __syncthreads();
  // output layer: y = W3 . H2 + b3 in feature order; dy = 2 (y - t) / nreal on
  // the real columns, 0 on the padding
  if (threadIdx.x < 16) {
    float y = b3;
#pragma unroll 16
    for (int f = 0; f < SUR_H; ++f) y += sw3[f] * sh2[f][col];
    s.yo[b] = y;
    if (s.y) {
      float d = 0.0f;
      if (real_row) {
        const float e = y - tgt;
        d = 2.0f * e / (float)s.nreal;
      }
      s.dy[b] = d;
      sdy[col] = d;
    }
  }
  if (!s.y) return;
  __syncthreads();
  // backward: dZ2 = W3 dy gelu'(Z2), dH1 = W2 dZ2, dZ1 = dH1 gelu'(Z1)
  float dz[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    dz[t] = w3[t] * sdy[col] * gelu_grad(z2[t]);
    s.dZ2[(size_t)(f0 + kq + t) * s.nb + b] = dz[t];
  }
  frag[1][wave][l] = pack4(dz[0], dz[1], dz[2], dz[3]);
  __syncthreads();
  acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)
    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w2b[kk], frag[1][kk][l], acc, 0, 0, 0);
#pragma unroll
  for (int t = 0; t < 4; ++t) s.dZ1[(size_t)(f0 + kq + t) * s.nb + b] = acc[t] * gelu_grad(z1[t]);
}

// Adam (Kingma & Ba 2015) on the FP32 master parameters.
struct AdamArgs {
  float *w, *m, *v;
  float lr, b1, b2, eps, c1, c2;
};
__device__ __forceinline__ void adam(const AdamArgs &a, int t, float gg) {
  const float mm = a.b1 * a.m[t] + (1.0f - a.b1) * gg;
  const float vv = a.b2 * a.v[t] + (1.0f - a.b2) * gg * gg;
  a.m[t] = mm;
  a.v[t] = vv;
  a.w[t] = a.w[t] - a.lr * (mm / a.c1) / (sqrtf(vv / a.c2) + a.eps);
}

// Parameter gradients of a batch, one role per block:
//   blocks 0 .. SUR_GB_W1-1   dW1[k][f] = sum_b X[b][k] dZ1[f][b], four 16 x 16
//                             tiles each (one per wave)
//   the next SUR_GB_W2        dW2[k][f] = sum_b H1[k][b] dZ2[f][b]
//   then one row sum each     dW3[f] = sum_b H2[f][b] dy[b], db3 = sum dy,
//                             db2[f] = sum dZ2[f], db1[f] = sum dZ1[f]
//   the last                  the loss: lossacc[q] = sum (y - t)^2 over columns
//                             256 q .. 256 q + 255, loss = scale sum lossacc
// ADAM: the update runs on the gradient where it is formed (nothing here
// reads the parameters); otherwise the gradients go to gr.
#define SUR_GB_W1 (SUR_K / 16)
#define SUR_GB_W2 4
#define SUR_GB_ROWS (3 * SUR_H + 1)
#define SUR_GB_ALL (SUR_GB_W1 + SUR_GB_W2 + SUR_GB_ROWS + 1)
// The products take SUR_GB_C columns at a time: the block gathers its 16
// inputs of those rows (64 bytes each) into LDS as BF16, all loads in flight
// together, and the waves issue SUR_GB_U loads of their other operand at once.
#define SUR_GB_C 512
#define SUR_GB_P (SUR_GB_C + 8)  // padded LDS row
#define SUR_GB_U 16
template <bool ADAM>
__global__ __launch_bounds__(256) void k_sur_grads(SurBatch s, AdamArgs a, float *__restrict__ gr,
                                                   float *__restrict__ lossacc, float scale, float *__restrict__ loss,
                                                   int drawn) {
  __shared__ float red[4];
  __shared__ __attribute__((aligned(16))) unsigned short sA[16 * SUR_GB_P];
  const int l = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
  const int col = l & 15, kq = 4 * (l >> 4), nb = s.nb;
  const int blk = (int)blockIdx.x;
  auto put = [&](int t, float v) {
    if (ADAM) adam(a, t, v);
    else gr[t] = v;
  };
  if (blk < SUR_GB_W1 + SUR_GB_W2) {
    const bool first = blk < SUR_GB_W1;
    const int m0 = (first ? blk : blk - SUR_GB_W1) * 16, n0 = wave * 16;
    const float *pb = (first ? s.dZ1 : s.dZ2) + (size_t)(n0 + col) * nb;
    const int t = (int)threadIdx.x, rq = t >> 2, cq = 4 * (t & 3);
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int c0 = 0; c0 < nb; c0 += SUR_GB_C) {
      const int cn = nb - c0 < SUR_GB_C ? nb - c0 : SUR_GB_C;
      // A(m, b): inputs m0 .. m0+15 (or rows of H1) of the columns, to sA[m][b]
      float4 v[SUR_GB_C / 64];
      if (first) {
        int row[SUR_GB_C / 64];
#pragma unroll
        for (int q = 0; q < SUR_GB_C / 64; ++q) {
          const int c = c0 + 64 * q + rq;
          row[q] = c < s.nreal ? (drawn ? s.row[c] : c) : -1;
        }
#pragma unroll
        for (int q = 0; q < SUR_GB_C / 64; ++q)
          v[q] = row[q] >= 0 ? *(const float4 *)(s.X + (size_t)row[q] * SUR_K + m0 + cq)
                             : float4{0.0f, 0.0f, 0.0f, 0.0f};
      } else {
        // thread (t & 15, t >> 4): row m0 + (t & 15), four columns at a time
#pragma unroll
        for (int q = 0; q < SUR_GB_C / 64; ++q) {
          const int c = 64 * q + 4 * (t >> 4);
          v[q] = c < cn ? *(const float4 *)(s.H1 + (size_t)(m0 + (t & 15)) * nb + c0 + c)
                        : float4{0.0f, 0.0f, 0.0f, 0.0f};
        }
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < SUR_GB_C / 64; ++q) {
        const bf16x4 p = pack4(v[q].x, v[q].y, v[q].z, v[q].w);
        if (first) {
#pragma unroll
          for (int j = 0; j < 4; ++j) sA[(cq + j) * SUR_GB_P + 64 * q + rq] = (unsigned short)p[j];
        } else {
          *(bf16x4 *)(sA + (t & 15) * SUR_GB_P + 64 * q + 4 * (t >> 4)) = p;
        }
      }
      __syncthreads();
      for (int k0 = 0; k0 < cn; k0 += 16 * SUR_GB_U) {
        float4 bv[SUR_GB_U];
#pragma unroll
        for (int q = 0; q < SUR_GB_U; ++q) {
          const int k = k0 + 16 * q < cn ? k0 + 16 * q : 0;  // past the end: any column, unused
          bv[q] = *(const float4 *)(pb + c0 + k + kq);
        }
#pragma unroll
        for (int q = 0; q < SUR_GB_U; ++q)
          if (k0 + 16 * q < cn)
            acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
                *(const bf16x4 *)(sA + col * SUR_GB_P + k0 + 16 * q + kq),
                pack4(bv[q].x, bv[q].y, bv[q].z, bv[q].w), acc, 0, 0, 0);
      }
    }
    const int off = first ? SUR_OFF_W1 : SUR_OFF_W2;
#pragma unroll
    for (int j = 0; j < 4; ++j) put(off + (m0 + kq + j) * SUR_H + n0 + col, acc[j]);
    return;
  }
  const int rs = blk - SUR_GB_W1 - SUR_GB_W2;
  if (rs < SUR_GB_ROWS) {
    const int f = rs < SUR_H ? rs : (rs - 1) % SUR_H;
    const float *m = rs < SUR_H ? s.H2 : (rs == SUR_H ? s.dy : (rs <= 2 * SUR_H ? s.dZ2 : s.dZ1));
    const int t = rs < SUR_H ? SUR_OFF_W3 + f
                             : (rs == SUR_H ? SUR_OFF_B3 : (rs <= 2 * SUR_H ? SUR_OFF_B2 + f : SUR_OFF_B1 + f));
    if (rs != SUR_H) m += (size_t)f * nb;
    float v = 0.0f;
    for (int b = (int)threadIdx.x; b < nb; b += 256) v += m[b] * (rs < SUR_H ? s.dy[b] : 1.0f);
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if (l == 0) red[wave] = v;
    __syncthreads();
    if (threadIdx.x == 0) put(t, red[0] + red[1] + red[2] + red[3]);
    return;
  }
  float sum = 0.0f;
  for (int q = 0; q * 256 < nb; ++q) {
    const int b = q * 256 + (int)threadIdx.x;
    float e2 = 0.0f;
    if (b < s.nreal) {
      const float e = s.yo[b] - s.y[drawn ? s.row[b] : b];
      e2 = e * e;
    }
    for (int off = 32; off > 0; off >>= 1) e2 += __shfl_down(e2, off, 64);
    if (l == 0) red[wave] = e2;
    __syncthreads();
    if (threadIdx.x == 0) {
      const float part = red[0] + red[1] + red[2] + red[3];
      lossacc[q] = part;
      sum += part;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0 && loss) *loss = sum * scale;
}

// ----------------------------------------------------------------------------
// inference over the interior
// ----------------------------------------------------------------------------
// BF16 copies of W1^T (64 x SUR_KP) and W2^T (64 x SUR_HP) for the LDS of the
// inference kernel.
__global__ void k_sur_pack(const float *__restrict__ w, unsigned short *__restrict__ w1t,
                           unsigned short *__restrict__ w2t) {
  const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (t < SUR_H * SUR_KP) {
    const int f = t / SUR_KP, kk = t % SUR_KP;
    w1t[t] = kk < SUR_K ? f2bf(w[SUR_OFF_W1 + kk * SUR_H + f]) : 0;
  }
  if (t < SUR_H * SUR_HP) {
    const int f = t / SUR_HP, kk = t % SUR_HP;
    w2t[t] = kk < SUR_H ? f2bf(w[SUR_OFF_W2 + kk * SUR_H + f]) : 0;
  }
}

// Inference over the interior with the features staged in LDS.  A block
// covers a tile of SIT_NW rows of SIT_WX cells (one row per wave) and
// marches in z over SIT_ZC planes, keeping the BF16 features of planes
// k-1, k, k+1 of the tile and its one-cell halo in a three-plane ring; each
// plane is read from HBM once per tile.  A wave computes its 64 cells as
// four 16-cell groups that share every W1^T fragment, so one LDS read of
// the weights feeds four MFMAs.  Per cell the layer-1 products accumulate
// over the 21 K steps in order, with the same BF16 operands as a per-cell
// gather.
#define SIT_WX 64
#define SIT_NW 8
#define SIT_ZC 8
#define SIT_RX (SIT_WX + 2)
#define SIT_RY (SIT_NW + 2)
#define SIT_PLANE (SIT_RX * SIT_RY * SUR_CH)  // bf16 elements of one staged plane
__global__ __launch_bounds__(64 * SIT_NW) void k_sur_infer_t(
    Geo g, const float *__restrict__ feat, const unsigned short *__restrict__ w1t,
    const unsigned short *__restrict__ w2t, const float *__restrict__ w, const real *__restrict__ E0,
    real *__restrict__ E1, double tfac, float y_scale) {
  __shared__ __attribute__((aligned(16))) unsigned short sW1[SUR_H * SUR_KP];
  __shared__ __attribute__((aligned(16))) unsigned short sW2[SUR_H * SUR_HP];
  __shared__ __attribute__((aligned(16))) unsigned short sF[3 * SIT_PLANE];
  __shared__ float sB1[SUR_H], sB2[SUR_H], sW3[SUR_H];
  for (int t = threadIdx.x; t < SUR_H * SUR_KP; t += blockDim.x) sW1[t] = w1t[t];
  for (int t = threadIdx.x; t < SUR_H * SUR_HP; t += blockDim.x) sW2[t] = w2t[t];
  for (int t = threadIdx.x; t < SUR_H; t += blockDim.x) {
    sB1[t] = w[SUR_OFF_B1 + t];
    sB2[t] = w[SUR_OFF_B2 + t];
    sW3[t] = w[SUR_OFF_W3 + t];
  }
  const float b3 = w[SUR_OFF_B3];
  const int l = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int col = l & 15, kq = 4 * (l >> 4);
  const int i0 = 1 + (int)blockIdx.x * SIT_WX, j0 = 1 + (int)blockIdx.y * SIT_NW, k0 = 1 + (int)blockIdx.z * SIT_ZC;
  const int k1 = k0 + SIT_ZC - 1 < g.nz ? k0 + SIT_ZC - 1 : g.nz;
  const int j = j0 + wave;
  // stage plane kk (0..n+1) of the tile and its halo into ring slot kk % 3;
  // halo points beyond n+1 (partial tiles) read cell n+1 and stay unused
  auto stage = [&](int kk) {
    unsigned short *P = sF + (kk % 3) * SIT_PLANE;
    for (int t = threadIdx.x; t < SIT_RX * SIT_RY * 3; t += blockDim.x) {
      const int cq = t % 3, r = t / 3;
      const int xx = r % SIT_RX, yy = r / SIT_RX;
      int ii = i0 - 1 + xx, jj = j0 - 1 + yy;
      ii = ii <= g.nx + 1 ? ii : g.nx + 1;
      jj = jj <= g.ny + 1 ? jj : g.ny + 1;
      const float4 x = *(const float4 *)(feat + (size_t)g.idx(ii, jj, kk) * SUR_CH + 4 * cq);
      *(bf16x4 *)(P + (yy * SIT_RX + xx) * SUR_CH + 4 * cq) = pack4(x.x, x.y, x.z, x.w);
    }
  };
  stage(k0 - 1);
  stage(k0);
  for (int k = k0; k <= k1; ++k) {
    stage(k + 1);
    __syncthreads();
    // layer 1: Z1^T (64 x 16 cells) per group = W1^T (64 x 336) . X^T
    f32x4 acc[4][4];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int cg = 0; cg < 4; ++cg) acc[mt][cg] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int st = 0; st < SUR_K / 16; ++st) {
      const int kb = st * 16 + kq;
      bf16x4 bop[4];
      if (kb < SUR_KREAL) {
        const int q = kb / SUR_CH, ch = kb % SUR_CH;
        const int dz = q / 9 - 1, dy = (q / 3) % 3 - 1, dx = q % 3 - 1;
        const unsigned short *P = sF + ((k + dz) % 3) * SIT_PLANE + ((wave + 1 + dy) * SIT_RX + 1 + dx) * SUR_CH + ch;
#pragma unroll
        for (int cg = 0; cg < 4; ++cg) bop[cg] = *(const bf16x4 *)(P + (16 * cg + col) * SUR_CH);
      } else {
#pragma unroll
        for (int cg = 0; cg < 4; ++cg) bop[cg] = bf16x4{0, 0, 0, 0};
      }
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        const bf16x4 aop = *(const bf16x4 *)(sW1 + (mt * 16 + col) * SUR_KP + kb);
#pragma unroll
        for (int cg = 0; cg < 4; ++cg)
          acc[mt][cg] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(aop, bop[cg], acc[mt][cg], 0, 0, 0);
      }
    }
#pragma unroll
    for (int cg = 0; cg < 4; ++cg) {
      bf16x4 h1[4];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        float hv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) hv[r] = gelu(acc[mt][cg][r] + sB1[mt * 16 + kq + r]);
        h1[mt] = pack4(hv[0], hv[1], hv[2], hv[3]);
      }
      // layer 2: Z2^T = W2^T (64 x 64) . H1^T (64 x 16)
      f32x4 acc2[4];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        acc2[mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          const bf16x4 aop = *(const bf16x4 *)(sW2 + (mt * 16 + col) * SUR_HP + kk * 16 + kq);
          acc2[mt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(aop, h1[kk], acc2[mt], 0, 0, 0);
        }
      }
      // layer 3 (FP32): y = W3 . GELU(Z2 + b2) + b3, summed over the 4 lane groups
      float part = 0.0f;
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int f = mt * 16 + kq + r;
          part += sW3[f] * gelu(acc2[mt][r] + sB2[f]);
        }
      part += __shfl_xor(part, 16, 64);
      part += __shfl_xor(part, 32, 64);
      const int i = i0 + 16 * cg + l;
      if (l < 16 && i <= g.nx && j <= g.ny) {
        const int c = g.idx(i, j, k);
        const double dT = (double)((part + b3) * y_scale);
        E1[c] = E0[c] + dT / tfac;
      }
    }
    __syncthreads();
  }
}

// Trapezoidal residual of a predicted super-step over the interior:
// partial sums of (E1 - E0 - trap)^2 and E0^2, with trap = dt/2 (L(E0) + L(E1)).
__global__ __launch_bounds__(BX * BY) void k_sur_residual(Geo g, const real *__restrict__ E0,
                                                          const real *__restrict__ E1,
                                                          const real *__restrict__ trap,
                                                          double *__restrict__ partial) {
  const Box b = {1, g.nx, 1, g.ny, 1, g.nz};
  PLANE_POS(b, i, j)
  const int k = 1 + (int)blockIdx.z;
  double v[2] = {0.0, 0.0};
  if (j <= g.ny && k <= g.nz) {
    const int c = g.idx(i, j, k);
    const double r = (E1[c] - E0[c]) - trap[c];
    v[0] = r * r;
    v[1] = E0[c] * E0[c];
  }
  const int ops[2] = {1, 1};
  block_reduce_store<2>(v, ops, partial);
}
