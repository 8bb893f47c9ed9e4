// mlp.hip -- per-particle pressure MLP for the PCISPH warm start, on BF16
// MFMA with FP32 accumulation (gfx950: v_mfma_f32_16x16x16_bf16).
//
// Network: 8 features -> 64 -> 64 -> 1, SiLU, 4,801 parameters.  FP32 master
// parameters, flat:  W1[64][8] @0, b1[64] @512, W2[64][64] @576, b2[64] @4672,
// W3[64] @4736, b3 @4800  (W[out][in]).  The layer-1 and layer-2 products
// and every weight-gradient product run on MFMA with BF16 operands; biases,
// activations and the 64-term output dot product are FP32.
//
// MFMA 16x16x16 fragment layouts (one wave, lane l, g = l / 16, r = l % 16):
//   A (16 x 16, [i][k])   a[j] = A[r][4g + j]
//   B (16 x 16, [k][n])   b[j] = B[4g + j][r]
//   D (16 x 16, [i][n])   d[j] = D[4g + j][r]
// A tile is 16 samples (particles).  Layer outputs come out in D layout
// (lane holds 4 samples of one unit); the next layer needs A layout (lane
// holds 4 units of one sample), so activations pass through a per-wave LDS
// tile.  In the backward pass the D-layout tiles are directly the A operand
// (dZ^T) and B operand (H) of the weight-gradient products, so those need no
// transpose.
#include <cmath>
#include <cstring>
#include <vector>

#include "psb_internal.h"
#include "mlp.h"

namespace psb {

typedef bf16x4_t bf16x4;
typedef float f32x4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even, on v_cvt_pk_bf16_f32 (an integer
// sequence with its NaN branch was a third of the training pass's
// instructions).
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t f2bf2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ uint16_t f2bf(float x) { return (uint16_t)f2bf2(x, 0.f); }
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ float sigm(float z) { return 1.0f / (1.0f + expf(-z)); }

__device__ __forceinline__ bf16x4 pack4(float a, float b, float c, float d) {
  return __builtin_bit_cast(bf16x4, make_uint2(f2bf2(a, b), f2bf2(c, d)));
}

__device__ __forceinline__ f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// ---- fragment packing of the FP32 master parameters --------------------------
// W1f[nt][l]: b[j] = W1[nt*16 + r][4g + j] (zero for inputs >= 8)
// W2f[kt][nt][l]: b[j] = W2[nt*16 + r][kt*16 + 4g + j]    (forward: Z2 = H1 W2^T)
// W2b[kt][nt][l]: b[j] = W2[kt*16 + 4g + j][nt*16 + r]    (backward: dH1 = dZ2 W2)
__global__ void k_mlp_pack(const float* __restrict__ w, MlpFrags f) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;   // 0 .. 36*64-1
  if (t >= 36 * 64) return;
  const int frag = t / 64, l = t % 64, g = l / 16, r = l % 16;
  const float* W1 = w + kOffW1;
  const float* W2 = w + kOffW2;
  float v[4];
  if (frag < 4) {
    const int nt = frag;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = 4 * g + j;
      v[j] = k < kIn ? W1[(nt * 16 + r) * kIn + k] : 0.f;
    }
    f.w1[frag * 64 + l] = pack4(v[0], v[1], v[2], v[3]);
  } else if (frag < 20) {
    const int kt = (frag - 4) / 4, nt = (frag - 4) % 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = W2[(nt * 16 + r) * kHid + kt * 16 + 4 * g + j];
    f.w2f[(frag - 4) * 64 + l] = pack4(v[0], v[1], v[2], v[3]);
  } else {
    const int kt = (frag - 20) / 4, nt = (frag - 20) % 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = W2[(kt * 16 + 4 * g + j) * kHid + nt * 16 + r];
    f.w2b[(frag - 20) * 64 + l] = pack4(v[0], v[1], v[2], v[3]);
  }
  if (t < kHid) f.w3[t] = bf2f(f2bf(w[kOffW3 + t]));
}

// Forward of one 16-sample tile.  a[j]: normalised input 4g + j of sample r
// of the tile (0 for padding).  Outputs in D layout: z1/h1, z2/h2
// [nt][j] = unit nt*16 + r of sample 4g + j; returns y for samples 4g + j in
// lanes with r == 0 (other lanes hold partial sums).
struct TileAct {
  f32x4 z1[4], z2[4], h1[4], h2[4];
  f32x4 s1[4], s2[4];   // sigmoid(z), read again by the backward pass
  float y[4];
};

__device__ __forceinline__ void tile_forward(const MlpFrags& f, const float* __restrict__ w,
                                             const float (&a)[4], uint16_t* lds, TileAct& t) {
  const int l = threadIdx.x & 63, g = l >> 4, r = l & 15;
  // layer 1: A1[r][4g+j] = a[j] = x[r][4g+j]
  const bf16x4 A1 = pack4(a[0], a[1], a[2], a[3]);
  const float* b1 = w + kOffB1;
  const float* b2 = w + kOffB2;
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    f32x4 z = mfma(A1, f.w1[nt * 64 + l], f32x4{0.f, 0.f, 0.f, 0.f});
    const float bias = b1[nt * 16 + r];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float zz = z[j] + bias;
      t.z1[nt][j] = zz;
      t.s1[nt][j] = sigm(zz);
      t.h1[nt][j] = zz * t.s1[nt][j];
      lds[(4 * g + j) * kLdsRow + nt * 16 + r] = f2bf(t.h1[nt][j]);
    }
  }
  __builtin_amdgcn_wave_barrier();
  // layer 2: A2[kt][r][4g+j] = h1[r][kt*16 + 4g + j]
  bf16x4 A2[4];
#pragma unroll
  for (int kt = 0; kt < 4; ++kt) {
    const uint16_t* src = lds + r * kLdsRow + kt * 16 + 4 * g;
    A2[kt] = bf16x4{(short)src[0], (short)src[1], (short)src[2], (short)src[3]};
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) z = mfma(A2[kt], f.w2f[(kt * 4 + nt) * 64 + l], z);
    const float bias = b2[nt * 16 + r];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float zz = z[j] + bias;
      t.z2[nt][j] = zz;
      t.s2[nt][j] = sigm(zz);
      t.h2[nt][j] = zz * t.s2[nt][j];
    }
  }
  // layer 3 (FP32 VALU): y[s] = sum_k h2[s][k] W3[k] + b3
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float s = 0.f;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) s = __builtin_fmaf(t.h2[nt][j], f.w3[nt * 16 + r], s);
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o, 16);
    t.y[j] = s + w[kOffB3];
  }
}

// Inference over n samples of a feature SoA [8][n]; y = max(0, out * pscale)
// written to pres[] and, when xw != nullptr, to the w lane of xw[].  With
// ids, samples whose id >= n_fluid (rigid-sphere boundary particles) get 0.
__global__ __launch_bounds__(256) void k_mlp_infer(const float* __restrict__ feat, uint32_t n,
                                                   const float* __restrict__ w, MlpFrags f,
                                                   MlpNorm nm, float* __restrict__ out,
                                                   float4* xw, float pscale, int clamp_relu,
                                                   const uint32_t* __restrict__ ids,
                                                   uint32_t n_fluid) {
  __shared__ uint16_t lds_all[4 * 16 * kLdsRow];
  const int wave = threadIdx.x >> 6;
  uint16_t* lds = lds_all + wave * 16 * kLdsRow;
  const uint64_t tile = (uint64_t)blockIdx.x * 4 + wave;
  const uint64_t p0 = tile * 16;
  if (p0 >= n) return;   // whole wave exits together
  const int l = threadIdx.x & 63, g = l >> 4, r = l & 15;
  float a[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    // clamped, so that the four loads go out together
    const int k = min(4 * g + j, kIn - 1);
    const uint64_t p = p0 + r < n ? p0 + r : n - 1u;
    const float v = (feat[(uint64_t)k * n + p] - nm.mu[k]) * nm.inv_sd[k];
    a[j] = (4 * g + j < kIn && p0 + r < n) ? v : 0.f;
  }
  TileAct t;
  tile_forward(f, w, a, lds, t);
  if (r == 0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint64_t p = p0 + 4 * g + j;
      if (p < n) {
        float v = t.y[j] * pscale;
        if (clamp_relu && v < 0.f) v = 0.f;
        if (ids && ids[p] >= n_fluid) v = 0.f;
        out[p] = v;
        if (xw) reinterpret_cast<float*>(xw)[4 * p + 3] = v;
      }
    }
  }
}

// Partial gradients: row b of part holds workgroup b's 4801 gradient entries
// (its four waves' sums added in wave order) and its loss sum at kOffLoss;
// k_mlp_update adds the rows in a fixed order, so a training run gives the
// same network every time.
constexpr int kOffLoss = kNumParams;
constexpr int kPartRow = kNumParams + 1;

// Forward + backward over a minibatch; each workgroup stores its gradient
// sums (and loss sum) into its row of part.  Samples idx[b0 .. b0 + nb) of the
// dataset (feature SoA [8][ns] + target[ns]); MSE on normalised targets.
__global__ __launch_bounds__(256) void k_mlp_train(const float* __restrict__ feat,
                                                   const float* __restrict__ target, uint64_t ns,
                                                   const uint32_t* __restrict__ idx, uint32_t nb,
                                                   const float* __restrict__ w, MlpFrags f,
                                                   MlpNorm nm, float* __restrict__ part) {
  __shared__ uint16_t lds_all[4 * 16 * kLdsRow];
  const int wave = threadIdx.x >> 6;
  uint16_t* lds = lds_all + wave * 16 * kLdsRow;
  const int l = threadIdx.x & 63, g = l >> 4, r = l & 15;
  const uint32_t ntiles = (nb + 15) / 16;
  const uint32_t wave_id = blockIdx.x * 4 + wave, nwaves = gridDim.x * 4;
  f32x4 gW2[4][4], gW1[4];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    gW1[a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < 4; ++b) gW2[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float gb1[4] = {0.f, 0.f, 0.f, 0.f}, gb2[4] = {0.f, 0.f, 0.f, 0.f}, gw3[4] = {0.f, 0.f, 0.f, 0.f};
  float gb3 = 0.f, lsum = 0.f;
  const float inv_b = 1.0f / (float)nb;
  for (uint32_t tile = wave_id; tile < ntiles; tile += nwaves) {
    const uint32_t s0 = tile * 16;
    // every load that depends on the sample indices goes out before the
    // forward pass (padding reads the last sample and is masked)
    const uint32_t sr = idx[min(s0 + r, nb - 1u)];
    uint32_t sj[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) sj[j] = idx[min(s0 + 4 * g + j, nb - 1u)];
    float xa[4], xb[4], tg[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = min(4 * g + j, kIn - 1), kr = min(r, kIn - 1);
      const float v = (feat[(uint64_t)k * ns + sr] - nm.mu[k]) * nm.inv_sd[k];
      xa[j] = (4 * g + j < kIn && s0 + r < nb) ? v : 0.f;
      const float u = (feat[(uint64_t)kr * ns + sj[j]] - nm.mu[kr]) * nm.inv_sd[kr];
      xb[j] = (r < kIn && s0 + 4 * g + j < nb) ? u : 0.f;
      tg[j] = target[sj[j]];
    }
    TileAct t;
    tile_forward(f, w, xa, lds, t);
    // dy for the 4 samples 4g + j, broadcast from lane 16g
    float dy[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float d = 0.f;
      if (s0 + 4 * g + j < nb) {
        const float e = t.y[j] - tg[j];
        d = 2.0f * e * inv_b;
        if (r == 0) lsum += e * e;
      }
      dy[j] = __shfl(d, 16 * g, 64);
    }
    // layer 3
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int j = 0; j < 4; ++j) gw3[nt] = __builtin_fmaf(t.h2[nt][j], dy[j], gw3[nt]);
    if (r == 0) gb3 += dy[0] + dy[1] + dy[2] + dy[3];
    // dZ2 = dy W3 * silu'(z2)   (D layout)
    f32x4 dz2[4];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      const float w3 = f.w3[nt * 16 + r];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float sg = t.s2[nt][j];
        const float dsilu = sg * (1.0f + t.z2[nt][j] * (1.0f - sg));
        dz2[nt][j] = dy[j] * w3 * dsilu;
        gb2[nt] += dz2[nt][j];
      }
    }
    // dW2[out][in] += sum_s dZ2[s][out] H1[s][in]:  A = dZ2^T (D tile), B = H1 (D tile)
    bf16x4 Ad[4], Bh[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      Ad[a] = pack4(dz2[a][0], dz2[a][1], dz2[a][2], dz2[a][3]);
      Bh[a] = pack4(t.h1[a][0], t.h1[a][1], t.h1[a][2], t.h1[a][3]);
    }
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int nk = 0; nk < 4; ++nk) gW2[mt][nk] = mfma(Ad[mt], Bh[nk], gW2[mt][nk]);
    // dH1 = dZ2 W2: dZ2 to A layout through LDS
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int j = 0; j < 4; ++j) lds[(4 * g + j) * kLdsRow + nt * 16 + r] = f2bf(dz2[nt][j]);
    __builtin_amdgcn_wave_barrier();
    bf16x4 A2[4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      const uint16_t* src = lds + r * kLdsRow + kt * 16 + 4 * g;
      A2[kt] = bf16x4{(short)src[0], (short)src[1], (short)src[2], (short)src[3]};
    }
    __builtin_amdgcn_wave_barrier();
    f32x4 dz1[4];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      f32x4 dh = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) dh = mfma(A2[kt], f.w2b[(kt * 4 + nt) * 64 + l], dh);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float sg = t.s1[nt][j];
        const float dsilu = sg * (1.0f + t.z1[nt][j] * (1.0f - sg));
        dz1[nt][j] = dh[j] * dsilu;
        gb1[nt] += dz1[nt][j];
      }
    }
    // dW1[out][in] += sum_s dZ1[s][out] X[s][in]:  A = dZ1^T (D tile), B[s][in] = x
    const bf16x4 Bx = pack4(xb[0], xb[1], xb[2], xb[3]);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
      gW1[mt] = mfma(pack4(dz1[mt][0], dz1[mt][1], dz1[mt][2], dz1[mt][3]), Bx, gW1[mt]);
  }
  // ---- flush: the waves add their sums into one LDS row, one after the
  // other, and the workgroup writes it out in full lines.  A row per wave was
  // 9.8 MB in 64-byte pieces for 512 waves, read back by the update: 23.8 us
  // for this pass and 9.1 for that, against 27.6 and 4.1. ----
  __shared__ float row[kPartRow];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    gb1[nt] += __shfl_xor(gb1[nt], 16, 64); gb1[nt] += __shfl_xor(gb1[nt], 32, 64);
    gb2[nt] += __shfl_xor(gb2[nt], 16, 64); gb2[nt] += __shfl_xor(gb2[nt], 32, 64);
    gw3[nt] += __shfl_xor(gw3[nt], 16, 64); gw3[nt] += __shfl_xor(gw3[nt], 32, 64);
  }
  gb3 += __shfl_xor(gb3, 16, 64); gb3 += __shfl_xor(gb3, 32, 64);
  lsum += __shfl_xor(lsum, 16, 64); lsum += __shfl_xor(lsum, 32, 64);
  for (uint32_t k = threadIdx.x; k < (uint32_t)kPartRow; k += blockDim.x) row[k] = 0.f;
  for (int turn = 0; turn < 4; ++turn) {
    __syncthreads();
    if (wave != turn) continue;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int out = mt * 16 + 4 * g + j;
        if (r < kIn) row[kOffW1 + out * kIn + r] += gW1[mt][j];
#pragma unroll
        for (int nk = 0; nk < 4; ++nk) row[kOffW2 + out * kHid + nk * 16 + r] += gW2[mt][nk][j];
      }
    }
    if (g == 0) {
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        row[kOffB1 + nt * 16 + r] += gb1[nt];
        row[kOffB2 + nt * 16 + r] += gb2[nt];
        row[kOffW3 + nt * 16 + r] += gw3[nt];
      }
    }
    if (l == 0) {
      row[kOffB3] += gb3;
      row[kOffLoss] += lsum;
    }
  }
  __syncthreads();
  float* dst = part + (size_t)blockIdx.x * kPartRow;
  for (uint32_t k = threadIdx.x; k < (uint32_t)kPartRow; k += blockDim.x) dst[k] = row[k];
}

// The rest of a training step in one launch: grad[k] += sum over the
// workgroups' rows of part[w][k], the loss sum, and with `apply` Adam (Kingma & Ba 2015) on
// the FP32 master parameters, the gradient zeroed and the parameter's BF16
// copies in the fragments rewritten.  Fixed order: row w goes to accumulator
// w % 8, the accumulators are added pairwise; the eight accumulators of a
// column are eight threads.  A batch of 8,192: 4.1 us, against 26 us for one
// thread per column (19 workgroups walking 512 rows) and 10 us for Adam and
// the fragments in launches of their own.
constexpr uint32_t kUpdateCols = 32;   // columns per workgroup (128-byte rows)
struct AdamArgs {
  int apply;
  float lr, b1, b2, eps, c1, c2;
};
__global__ __launch_bounds__(8 * kUpdateCols) void k_mlp_update(
    const float* __restrict__ part, uint32_t rows, float* __restrict__ grad, float* loss,
    float* __restrict__ w, float* __restrict__ m1, float* __restrict__ m2, MlpFrags f, AdamArgs a) {
  __shared__ float acc8[8][kUpdateCols];
  const uint32_t u = threadIdx.x / kUpdateCols, col = threadIdx.x % kUpdateCols;
  const uint32_t k = blockIdx.x * kUpdateCols + col;
  float acc = 0.f;
  if (k < (uint32_t)kPartRow) {
    const float* src = part + (size_t)u * kPartRow + k;
    const size_t step = 8 * (size_t)kPartRow;
    uint32_t r = u;
    for (; r + 56u < rows; r += 64u, src += 8 * step) {   // 8 rows of this accumulator in flight
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = src[j * step];
#pragma unroll
      for (int j = 0; j < 8; ++j) acc += v[j];
    }
    for (; r < rows; r += 8u, src += step) acc += *src;
  }
  acc8[u][col] = acc;
  __syncthreads();
  if (u != 0u || k >= (uint32_t)kPartRow) return;
  const float sum = ((acc8[0][col] + acc8[1][col]) + (acc8[2][col] + acc8[3][col])) +
                    ((acc8[4][col] + acc8[5][col]) + (acc8[6][col] + acc8[7][col]));
  if (k == (uint32_t)kOffLoss) { *loss = sum; return; }
  const float gr = grad[k] + sum;
  if (!a.apply) { grad[k] = gr; return; }
  const float m = a.b1 * m1[k] + (1.0f - a.b1) * gr;
  const float v = a.b2 * m2[k] + (1.0f - a.b2) * gr * gr;
  m1[k] = m;
  m2[k] = v;
  const float wn = w[k] - a.lr * (m / a.c1) / (sqrtf(v / a.c2) + a.eps);
  w[k] = wn;
  grad[k] = 0.f;
  const uint16_t h = f2bf(wn);
  if (k < (uint32_t)kOffB1) {
    const uint32_t o = k / kIn, i = k % kIn;
    reinterpret_cast<uint16_t*>(f.w1)[((o >> 4) * 64u + (i >> 2) * 16u + (o & 15u)) * 4u + (i & 3u)] = h;
  } else if (k >= (uint32_t)kOffW2 && k < (uint32_t)kOffB2) {
    const uint32_t o = (k - kOffW2) / kHid, i = (k - kOffW2) % kHid;
    // element (o, i) as W2[row][4g + j] of tile (tr, tk): see k_mlp_pack
    auto at = [](uint32_t row, uint32_t kk) {
      return (((kk >> 4) * 4u + (row >> 4)) * 64u + (kk >> 2 & 3u) * 16u + (row & 15u)) * 4u + (kk & 3u);
    };
    reinterpret_cast<uint16_t*>(f.w2f)[at(o, i)] = h;
    reinterpret_cast<uint16_t*>(f.w2b)[at(i, o)] = h;
  } else if (k >= (uint32_t)kOffW3 && k < (uint32_t)kOffB3) {
    f.w3[k - kOffW3] = bf2f(h);
  }
}

}  // namespace psb

using namespace psb;

struct psb_mlp_s {
  psb_context ctx = nullptr;
  float* w = nullptr;      // [kNumParams] FP32 master
  float* grad = nullptr;   // [kNumParams]
  float* m1 = nullptr;
  float* m2 = nullptr;
  float* h_loss = nullptr; // host-mapped: the last training step's loss sum
  float* d_loss = nullptr;
  float* part = nullptr;   // per-workgroup gradient rows of a training step
  uint32_t part_rows = 0;
  MlpFrags frags{};
  void* frag_mem = nullptr;
  MlpNorm norm{};
  float pscale = 1.f;
  int64_t adam_t = 0;
};

namespace psb {

psb_status mlp_pack(psb_mlp m) {
  hipLaunchKernelGGL(k_mlp_pack, dim3((36 * 64 + 255) / 256), dim3(256), 0, m->ctx->stream, m->w,
                     m->frags);
  PSB_HIP(hipGetLastError());
  return PSB_OK;
}

psb_status mlp_infer(psb_mlp m, const float* feat, uint32_t n, float* out, float4* xw, int relu,
                     float scale, hipStream_t s, const uint32_t* ids, uint32_t n_fluid) {
  if (!n) return PSB_OK;
  const uint32_t tiles = (n + 15) / 16;
  hipLaunchKernelGGL(k_mlp_infer, dim3((tiles + 3) / 4), dim3(256), 0, s, feat, n, m->w, m->frags,
                     m->norm, out, xw, scale, relu, ids, n_fluid);
  PSB_HIP(hipGetLastError());
  return PSB_OK;
}

float mlp_pscale(psb_mlp m) { return m->pscale; }

}  // namespace psb

extern "C" {

psb_status psb_mlp_create(psb_context ctx, uint64_t seed, psb_mlp* out) {
  PSB_ARG(ctx && out, "null argument");
  PSB_HIP(hipSetDevice(ctx->device));
  psb_mlp m = new psb_mlp_s();
  m->ctx = ctx;
  auto fail = [&](hipError_t e) { psb_mlp_destroy(m); return hip_fail(e, "mlp alloc", __FILE__, __LINE__); };
  hipError_t e;
  if ((e = hipMalloc(&m->w, 4 * kNumParams)) != hipSuccess) return fail(e);
  if ((e = hipMalloc(&m->grad, 4 * kNumParams)) != hipSuccess) return fail(e);
  if ((e = hipMalloc(&m->m1, 4 * kNumParams)) != hipSuccess) return fail(e);
  if ((e = hipMalloc(&m->m2, 4 * kNumParams)) != hipSuccess) return fail(e);
  if ((e = take_line(ctx, (void**)&m->h_loss, (void**)&m->d_loss)) != hipSuccess) return fail(e);
  const size_t fb = sizeof(bf16x4) * 64 * 36 + 4 * kHid;
  if ((e = hipMalloc(&m->frag_mem, fb)) != hipSuccess) return fail(e);
  bf16x4* fm = (bf16x4*)m->frag_mem;
  m->frags.w1 = fm;
  m->frags.w2f = fm + 4 * 64;
  m->frags.w2b = fm + 20 * 64;
  m->frags.w3 = (float*)(fm + 36 * 64);
  for (int k = 0; k < kIn; ++k) { m->norm.mu[k] = 0.f; m->norm.inv_sd[k] = 1.f; }
  // He-uniform initialisation from a splitmix64 stream (deterministic)
  std::vector<float> w(kNumParams, 0.f);
  uint64_t st = seed ? seed : 0x9e3779b97f4a7c15ull;
  auto next = [&]() {
    uint64_t z = (st += 0x9e3779b97f4a7c15ull);
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    z ^= z >> 31;
    return (double)(z >> 11) * (1.0 / 9007199254740992.0);
  };
  auto fill = [&](int off, int cnt, int fan_in) {
    const double a = std::sqrt(6.0 / fan_in);
    for (int i = 0; i < cnt; ++i) w[off + i] = (float)((2.0 * next() - 1.0) * a);
  };
  fill(kOffW1, kHid * kIn, kIn);
  fill(kOffW2, kHid * kHid, kHid);
  fill(kOffW3, kHid, kHid);
  return psb_mlp_set_params(m, w.data(), kNumParams) == PSB_OK ? (*out = m, PSB_OK)
                                                               : (psb_mlp_destroy(m), PSB_ERR_HIP);
}

psb_status psb_mlp_destroy(psb_mlp m) {
  if (!m) return PSB_OK;
  hipSetDevice(m->ctx->device);
  hipStreamSynchronize(m->ctx->stream);
  hipFree(m->w); hipFree(m->grad); hipFree(m->m1); hipFree(m->m2);
  if (m->h_loss) give_line(m->ctx, m->h_loss);
  hipFree(m->frag_mem);
  if (m->part) hipFree(m->part);
  delete m;
  return PSB_OK;
}

int32_t psb_mlp_num_params(void) { return kNumParams; }

psb_status psb_mlp_set_params(psb_mlp m, const float* host_w, int32_t count) {
  PSB_ARG(m && host_w && count == kNumParams, "psb_mlp_set_params: need 4801 parameters");
  hipStream_t s = m->ctx->stream;
  PSB_HIP(hipMemcpyAsync(m->w, host_w, 4 * kNumParams, hipMemcpyHostToDevice, s));
  PSB_HIP(hipMemsetAsync(m->grad, 0, 4 * kNumParams, s));
  PSB_HIP(hipMemsetAsync(m->m1, 0, 4 * kNumParams, s));
  PSB_HIP(hipMemsetAsync(m->m2, 0, 4 * kNumParams, s));
  m->adam_t = 0;
  PSB_TRY(mlp_pack(m));
  PSB_HIP(hipStreamSynchronize(s));
  return PSB_OK;
}

psb_status psb_mlp_get_params(psb_mlp m, float* host_w, int32_t count) {
  PSB_ARG(m && host_w && count == kNumParams, "psb_mlp_get_params: need 4801 parameters");
  PSB_HIP(hipMemcpyAsync(host_w, m->w, 4 * kNumParams, hipMemcpyDeviceToHost, m->ctx->stream));
  PSB_HIP(hipStreamSynchronize(m->ctx->stream));
  return PSB_OK;
}

psb_status psb_mlp_set_normalization(psb_mlp m, const float mean[8], const float stddev[8],
                                     float pressure_scale) {
  PSB_ARG(m && mean && stddev && pressure_scale > 0.f, "bad normalisation");
  for (int k = 0; k < kIn; ++k) {
    PSB_ARG(stddev[k] > 0.f, "stddev must be > 0");
    m->norm.mu[k] = mean[k];
    m->norm.inv_sd[k] = 1.0f / stddev[k];
  }
  m->pscale = pressure_scale;
  return PSB_OK;
}

psb_status psb_mlp_forward(psb_mlp m, const float* features, uint32_t n, float* out) {
  PSB_ARG(m && (n == 0 || (features && out)), "null argument");
  PSB_TRY(mlp_infer(m, features, n, out, nullptr, 0, 1.0f, m->ctx->stream));
  return PSB_OK;
}

psb_status psb_mlp_train_step(psb_mlp m, const float* features, const float* targets,
                              uint64_t num_samples, const uint32_t* batch_idx, uint32_t batch,
                              float lr, int32_t apply_adam, float* loss_out) {
  PSB_ARG(m && features && targets && batch_idx && batch > 0, "null argument");
  hipStream_t s = m->ctx->stream;
  const uint32_t tiles = (batch + 15) / 16;
  uint32_t blocks = (tiles + 3) / 4;
  if (blocks > 512) blocks = 512;
  const uint32_t rows = blocks;
  if (rows > m->part_rows) {
    PSB_HIP(hipStreamSynchronize(s));
    if (m->part) PSB_HIP(hipFree(m->part));
    m->part = nullptr;
    m->part_rows = 0;
    PSB_HIP(hipMalloc((void**)&m->part, (size_t)rows * kPartRow * sizeof(float)));
    m->part_rows = rows;
  }
  hipLaunchKernelGGL(k_mlp_train, dim3(blocks), dim3(256), 0, s, features, targets, num_samples,
                     batch_idx, batch, m->w, m->frags, m->norm, m->part);
  PSB_HIP(hipGetLastError());
  AdamArgs a{};
  if (apply_adam) {
    m->adam_t += 1;
    a.apply = 1;
    a.lr = lr;
    a.b1 = 0.9f;
    a.b2 = 0.999f;
    a.eps = 1e-8f;
    a.c1 = (float)(1.0 - std::pow(0.9, (double)m->adam_t));
    a.c2 = (float)(1.0 - std::pow(0.999, (double)m->adam_t));
  }
  hipLaunchKernelGGL(k_mlp_update, dim3((kPartRow + kUpdateCols - 1) / kUpdateCols),
                     dim3(8 * kUpdateCols), 0, s, m->part, rows, m->grad, m->d_loss, m->w, m->m1,
                     m->m2, m->frags, a);
  PSB_HIP(hipGetLastError());
  if (loss_out) {
    PSB_HIP(hipStreamSynchronize(s));
    *loss_out = *(volatile float*)m->h_loss / (float)batch;
  }
  return PSB_OK;
}

psb_status psb_mlp_get_grad(psb_mlp m, float* host_grad, int32_t count) {
  PSB_ARG(m && host_grad && count == kNumParams, "need 4801 entries");
  PSB_HIP(hipMemcpyAsync(host_grad, m->grad, 4 * kNumParams, hipMemcpyDeviceToHost, m->ctx->stream));
  PSB_HIP(hipStreamSynchronize(m->ctx->stream));
  return PSB_OK;
}

psb_status psb_mlp_zero_grad(psb_mlp m) {
  PSB_ARG(m, "null mlp");
  PSB_HIP(hipMemsetAsync(m->grad, 0, 4 * kNumParams, m->ctx->stream));
  return PSB_OK;
}

}  // extern "C"
