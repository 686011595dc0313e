// Training and inference kernels of the learned eddy-viscosity closure's
// network (dh_mlp_dev.h): operand packing, batched inference, the forward
// and backward pass of a batch with the weight gradients as BF16 MFMA GEMMs
// over its samples, the reduction of per-block partial gradients, and Adam.
// No counterpart in the reference (its LES has no learned model).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "dh_internal.h"
#include "dh_mlp_dev.h"

namespace dh {

// Packs the FP32 parameters into the BF16 operand order of dh_mlp_dev.h.
// One thread per (array, lane) writes the lane's 8 values.
__global__ void k_mlp_pack(const float *__restrict__ P, bf16x8 *__restrict__ pk) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= kPAll) return;
  const int lane = t & 63, g = lane >> 4, c = lane & 15;
  if (t >= kPBias) {  // biases and w4 in the result-tile layout
    const int r = (t - kPBias) >> 6, layer = r >> 2, mt = r & 3;  // layer 3: w4
    const int off = (layer == 0) ? kOB1 : (layer == 1) ? kOB2 : (layer == 2) ? kOB3 : kOW4;
    f32x4 b;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v = P[off + 16 * mt + 4 * g + i];
      b[i] = (layer == 3) ? (float)(__bf16)v : v;
    }
    reinterpret_cast<f32x4 *>(pk)[t] = b;
    return;
  }
  bf16x8 v;
  if (t < kPA2) {  // A1[mt][lane]: W1[8 g + j][16 mt + c]
    const int mt = t >> 6;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (__bf16)P[kOW1 + (8 * g + j) * kMlpH + 16 * mt + c];
  } else if (t < kPA4) {  // A2, A3 [mt][kb][lane]: W[u(kb,g,j)][16 mt + c]
    const int base = (t < kPA3) ? kOW2 : kOW3, r = (t - ((t < kPA3) ? kPA2 : kPA3)) >> 6;
    const int mt = r >> 1, kb = r & 1;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (__bf16)P[base + mlp_unit(kb, g, j) * kMlpH + 16 * mt + c];
  } else if (t < kPB2) {  // A4[kb][lane]: row 0 is w4
    const int kb = (t - kPA4) >> 6;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (__bf16)(c == 0 ? P[kOW4 + mlp_unit(kb, g, j)] : 0.0f);
  } else {  // B2, B3 [mt][kb][lane]: W[16 mt + c][u(kb,g,j)] (untransposed)
    const int base = (t < kPB3) ? kOW2 : kOW3, r = (t - ((t < kPB3) ? kPB2 : kPB3)) >> 6;
    const int mt = r >> 1, kb = r & 1;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (__bf16)P[base + (16 * mt + c) * kMlpH + mlp_unit(kb, g, j)];
  }
  pk[t] = v;
}

// layer-1 operand of this lane: features 8 g + j (< nin) of sample n, from a
// feature-major array x[f * ld + n] (zero for n >= N)
// (only lane group 0 holds inputs; ld * 8 < 2^31, checked by the host)
__device__ __forceinline__ bf16x8 load_x(const float *__restrict__ x, long long ld, long long n, long long N, int nin) {
  const int g = (threadIdx.x & 63) >> 4;
  bf16x8 v;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = (__bf16)0.0f;
  if (g == 0 && n < N) {
    const float *xn = x + n;
    const int ldi = (int)ld;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j < nin) v[j] = (__bf16)xn[j * ldi];
  }
  return v;
}

// out[n] = scale * softplus(y(x_n)), x feature-major [6][ld]
__global__ void __launch_bounds__(256) k_mlp_infer(const bf16x8 *__restrict__ pk, const float *__restrict__ P,
                                                 const float *__restrict__ x, long long ld, long long N,
                                                 float scale, float *__restrict__ out) {
  const int lane = threadIdx.x & 63;
  const long long wave = ((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const long long nw = ((long long)gridDim.x * blockDim.x) >> 6;
  MlpRegs r;
  mlp_load_regs(pk, r);
  const float b4 = P[kOB4];
  for (long long n0 = wave * 16; n0 < N; n0 += nw * 16) {
    const long long n = n0 + (lane & 15);
    const bf16x8 xb = load_x(x, ld, n, N, kMlpIn);
    const float y = mlp_forward_regs(r, b4, xb);
    if (lane < 16 && n < N) out[n] = scale * softplus(y);
  }
}

// Loss, forward and backward pass and the weight gradients of a batch, one
// launch.  Loss: sum_n (softplus(y_n) - t_n)^2 / N.  A block of four waves
// takes 64 samples at a time, 16 per wave through the network and back; the
// layer inputs H0 (features), H1..H3, dL/dy and the pre-activation gradients
// dZ1..dZ3 go to LDS as BF16 rows of the tile's samples, which is the
// transpose the gradient products need: 16x16x32 BF16 MFMAs with the samples
// as K (lane l reads 8 consecutive samples of one row for A and for B),
//   dW[in][out] = sum_n Hin[in][n] dZ[out][n],  wave w the columns
//   out = 16 w + l % 16 of every layer (layer 1 has one row tile, inputs
//   0..15, of which 0..7 are non-zero), the bias gradients sum_n dZ[out][n]
//   from an A operand of ones, dW4[u] = sum_n H3[u][n] dy[n] for the rows
//   16 w + l % 16 (dy in column 0 of B) and db4 = sum_n dy[n] (wave 0).
// A block keeps its sums in registers over its tiles and writes them once,
// in the parameter vector's layout, to part[block][kPartLd] (rows 8..31 of
// W1, which have no inputs, are left out; the block's loss at kMlpNP).
//
// What bounds it: the chain of layers (MFMA, GELU, conversion, next MFMA) at
// two waves per SIMD; 800 B of activations per sample stay in LDS.  With the
// activations in device memory between a pass kernel and a product kernel of
// one wave per 1024 samples and layer (64 waves at 16384 samples), a step of
// 16384 samples took 100 us, 47 of them in the products and 23 in the sum
// over 512 partial losses by one thread; this way the whole step (this
// launch, the sum over blocks 4.5 us, the update 2.4 us) takes 21 us.
constexpr int kTrThreads = 256, kTrTile = 64;
constexpr int kTrLd = kTrTile + 8;      // row stride in LDS (BF16 values): rows start on different banks
constexpr int kRH0 = 0, kRH1 = 8, kRD1 = kRH1 + 3 * kMlpH, kRDY = kRD1 + 3 * kMlpH, kTrRows = kRDY + 1;
constexpr int kPartLd = (kMlpNP + 1 + 3) / 4 * 4;  // floats per block of partial sums

__global__ void __launch_bounds__(kTrThreads, 2) k_mlp_train(const bf16x8 *pk, const float *P,
                                                           const float *__restrict__ x, const float *__restrict__ t,
                                                           long long N, float inv_n, float *__restrict__ part) {
  __shared__ alignas(bf16x8) __bf16 act[kTrRows * kTrLd];
  static_assert(__alignof__(act) >= alignof(bf16x8) && kTrLd * sizeof(__bf16) % alignof(bf16x8) == 0,
                "a row is read in pieces of 8 values");
  __shared__ float wloss[kTrThreads / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 aw1 = zero, aw2[4], aw3[4], ab[3], aw4 = zero, ab4 = zero;
#pragma unroll
  for (int i = 0; i < 4; ++i) aw2[i] = aw3[i] = zero;
#pragma unroll
  for (int i = 0; i < 3; ++i) ab[i] = zero;
  bf16x8 ones, none;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    ones[j] = (__bf16)1.0f;
    none[j] = (__bf16)0.0f;
  }
  float sloss = 0.f;
  const float b4 = P[kOB4];
  const int col = 16 * w + c;  // this lane's sample in the tile
  const long long nt = (N + kTrTile - 1) / kTrTile;
  for (long long tile = blockIdx.x; tile < nt; tile += gridDim.x) {
    // operands re-read each pass: neither they nor their addresses (two
    // registers each) are held across it
    const bf16x8 *pl = pk + lane;
    asm volatile("" : "+v"(pl)::"memory");
    const long long n = tile * kTrTile + col;
    const bool live = n < N;
    const bf16x8 xb = load_x(x, N, n, N, kMlpIn);
    auto put = [&](int row0, int u, float v) { act[(row0 + u) * kTrLd + col] = (__bf16)v; };
    if (g == 0) {
#pragma unroll
      for (int j = 0; j < 8; ++j) act[(kRH0 + j) * kTrLd + col] = xb[j];
    }
    // forward, layer by layer; of a layer only GELU'(Z) stays in registers
    // (its GELU(Z) in LDS, and as the next layer's operand)
    f32x4 gp[3][4], h[4];
    auto activate = [&](f32x4 (&z)[4], int layer) {
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float zi = z[mt][i], s = gelu_s(zi);
          h[mt][i] = zi * s;
          gp[layer][mt][i] = gelu_grad(zi, s);
          put(kRH1 + layer * kMlpH, 16 * mt + 4 * g + i, h[mt][i]);
        }
      // a layer's operands are not loaded ahead of the layer before it: all
      // 34 together with the sums would spill
      asm volatile("" ::: "memory");
    };
    const f32x4 *pb = reinterpret_cast<const f32x4 *>(pl) + kPBias;
    {
      const bf16x8 b[1] = {xb};
      f32x4 z[4];
      mlp_layer<1>(pl + kPA1, b, pb, z);
      activate(z, 0);
    }
#pragma unroll
    for (int layer = 1; layer < 3; ++layer) {
      const bf16x8 b[2] = {pack_b(h, 0), pack_b(h, 1)};
      f32x4 z[4];
      mlp_layer<2>(pl + (layer == 1 ? kPA2 : kPA3), b, pb + 4 * layer * 64, z);
      activate(z, layer);
    }
    f32x4 yd = zero;
    yd = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pl[kPA4], pack_b(h, 0), yd, 0, 0, 0);
    yd = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pl[kPA4 + 64], pack_b(h, 1), yd, 0, 0, 0);
    const float y = yd[0] + b4;
    asm volatile("" ::: "memory");  // nor the backward operands
    float dy = 0.f;  // zero for samples beyond N, and with it every gradient of theirs
    if (lane < 16) {
      if (live) {
        const float r = softplus(y) - t[n];
        sloss += r * r;
        dy = 2.0f * r * sigmoid(y) * inv_n;
      }
      act[kRDY * kTrLd + col] = (__bf16)dy;
    }
    const float dys = __shfl(dy, c);  // this lane's sample
    // dZ3 = dy w4 GELU'(Z3) (w4 rounded as the forward pass used it), then
    // dH2 = W3 dZ3^T, dZ2 = dH2 GELU'(Z2); dH1 = W2 dZ2^T, dZ1 = dH1 GELU'(Z1)
    f32x4 d[4];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const f32x4 w4 = reinterpret_cast<const f32x4 *>(pl)[kPW4 + mt * 64];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        d[mt][i] = dys * w4[i] * gp[2][mt][i];
        put(kRD1 + 2 * kMlpH, 16 * mt + 4 * g + i, d[mt][i]);
      }
    }
#pragma unroll
    for (int layer = 1; layer >= 0; --layer) {
      asm volatile("" ::: "memory");
      const bf16x8 b[2] = {pack_b(d, 0), pack_b(d, 1)};
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        f32x4 q = zero;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
          q = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pl[(layer ? kPB3 : kPB2) + (mt * 2 + kb) * 64], b[kb], q, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          d[mt][i] = q[i] * gp[layer][mt][i];
          put(kRD1 + layer * kMlpH, 16 * mt + 4 * g + i, d[mt][i]);
        }
      }
    }
    __syncthreads();
    auto row = [&](int r, int k0) { return *reinterpret_cast<const bf16x8 *>(&act[r * kTrLd + k0 + 8 * g]); };
#pragma unroll 1
    for (int k0 = 0; k0 < kTrTile; k0 += 32) {
      const bf16x8 d1b = row(kRD1 + col, k0), d2b = row(kRD1 + kMlpH + col, k0), d3b = row(kRD1 + 2 * kMlpH + col, k0);
      const bf16x8 dyb = (c == 0) ? row(kRDY, k0) : none;
      const bf16x8 h0 = (c < 8) ? row(kRH0 + c, k0) : none;
      aw1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h0, d1b, aw1, 0, 0, 0);
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        aw2[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(row(kRH1 + 16 * mt + c, k0), d2b, aw2[mt], 0, 0, 0);
        aw3[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(row(kRH1 + kMlpH + 16 * mt + c, k0), d3b, aw3[mt], 0, 0, 0);
      }
      ab[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, d1b, ab[0], 0, 0, 0);
      ab[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, d2b, ab[1], 0, 0, 0);
      ab[2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, d3b, ab[2], 0, 0, 0);
      aw4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(row(kRH1 + 2 * kMlpH + col, k0), dyb, aw4, 0, 0, 0);
      if (w == 0) ab4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, dyb, ab4, 0, 0, 0);
    }
    __syncthreads();  // the next tile's rows go over these
  }
  // result tiles: lane l holds rows 4 g + i of column c
  float *o = part + (long long)blockIdx.x * kPartLd;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (g < 2) o[kOW1 + (4 * g + i) * kMlpH + col] = aw1[i];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      o[kOW2 + (16 * mt + 4 * g + i) * kMlpH + col] = aw2[mt][i];
      o[kOW3 + (16 * mt + 4 * g + i) * kMlpH + col] = aw3[mt][i];
    }
    if (c == 0) o[kOW4 + 16 * w + 4 * g + i] = aw4[i];
  }
  if (g == 0) {  // every row of a ones tile holds the column sums
    o[kOB1 + col] = ab[0][0];
    o[kOB2 + col] = ab[1][0];
    o[kOB3 + col] = ab[2][0];
  }
  if (threadIdx.x == 0) o[kOB4] = ab4[0];
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) sloss += __shfl_xor(sloss, s);
  if (lane == 0) wloss[w] = sloss * inv_n;  // the loss is the mean over the batch
  __syncthreads();
  if (threadIdx.x == 0) o[kMlpNP] = (wloss[0] + wloss[1]) + (wloss[2] + wloss[3]);
}

// grad[p] = the sum of the blocks' partial sums (rows 8..31 of W1 are zero:
// their inputs are zero); loss = the sum of their parts of the batch mean.
// A block takes 64 values, its four waves every fourth partial sum each, so
// that 165 blocks of four waves read the partial sums (42 KB per block of
// k_mlp_train) with eight loads in flight per lane.
__global__ void __launch_bounds__(256) k_mlp_reduce(const float *__restrict__ part, int nblk, float *__restrict__ grad,
                                                  float *__restrict__ loss) {
  __shared__ float sm[4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, p = blockIdx.x * 64 + lane;
  const bool padding = p >= 8 * kMlpH && p < kOB1;
  float a = 0.f;
  if (p <= kMlpNP && !padding) {
#pragma unroll 8
    for (int k = w; k < nblk; k += 4) a += part[(long long)k * kPartLd + p];
  }
  sm[w][lane] = a;
  __syncthreads();
  if (w != 0 || p > kMlpNP) return;
  a = (sm[0][lane] + sm[1][lane]) + (sm[2][lane] + sm[3][lane]);
  if (p == kMlpNP)
    *loss = a;
  else
    grad[p] = a;
}

// Adam (Kingma & Ba 2015) on the FP32 parameters; c1 = 1 - beta1^t,
// c2 = 1 - beta2^t come from the host.  Each thread also writes its new
// parameter to every place k_mlp_pack would put it (the zero rows of the
// output layer's operand included), so the update is one launch; a second
// one for the packing took 4.8 us and the gap before it, at 5 us a launch
// for 42 KB of parameters.
__global__ void __launch_bounds__(64) k_mlp_adam_pack(float *__restrict__ P, float *__restrict__ m,
                                                    float *__restrict__ v, const float *__restrict__ grad, float lr,
                                                    float b1, float b2, float eps, float c1, float c2,
                                                    bf16x8 *__restrict__ pk) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= kMlpNP) return;
  const float gr = grad[p];
  const float mm = b1 * m[p] + (1.f - b1) * gr, vv = b2 * v[p] + (1.f - b2) * gr * gr;
  m[p] = mm;
  v[p] = vv;
  const float w = P[p] - lr * (mm / c1) / (sqrtf(vv / c2) + eps);
  P[p] = w;
  __bf16 *q = reinterpret_cast<__bf16 *>(pk);
  float *qf = reinterpret_cast<float *>(pk);
  const __bf16 wb = (__bf16)w;
  // lane and element of unit u (mlp_unit's inverse): K block u / 32, lane
  // group (u / 4) % 4, element 4 ((u / 16) % 2) + u % 4
  auto unit = [](int u, int c) { return ((u >> 5) * 64 + 16 * ((u >> 2) & 3) + c) * 8 + 4 * ((u >> 4) & 1) + (u & 3); };
  auto tile = [&](int base, int u, float val) {  // result-tile layout, the 16 lanes of the unit's group
#pragma unroll
    for (int c = 0; c < 16; ++c) qf[(base + (u >> 4) * 64 + 16 * ((u >> 2) & 3) + c) * 4 + (u & 3)] = val;
  };
  auto hidden = [&](int pa, int pb, int r) {  // W[in][out] as A (transposed) and B operands
    const int in = r / kMlpH, out = r % kMlpH;
    q[(pa + (out >> 4) * 128) * 8 + unit(in, out & 15)] = wb;
    q[(pb + (in >> 4) * 128) * 8 + unit(out, in & 15)] = wb;
  };
  if (p < kOB1) {
    const int in = p / kMlpH, out = p % kMlpH;
    q[(kPA1 + (out >> 4) * 64 + 16 * (in >> 3) + (out & 15)) * 8 + (in & 7)] = wb;
  } else if (p < kOW2) {
    tile(kPBias, p - kOB1, w);
  } else if (p < kOB2) {
    hidden(kPA2, kPB2, p - kOW2);
  } else if (p < kOW3) {
    tile(kPBias + 4 * 64, p - kOB2, w);
  } else if (p < kOB3) {
    hidden(kPA3, kPB3, p - kOW3);
  } else if (p < kOW4) {
    tile(kPBias + 8 * 64, p - kOB3, w);
  } else if (p < kOB4) {
    const int u = p - kOW4;
#pragma unroll
    for (int c = 0; c < 16; ++c) q[kPA4 * 8 + unit(u, c)] = c == 0 ? wb : (__bf16)0.0f;
    tile(kPW4, u, (float)wb);
  }
}

hipError_t launch_mlp_pack(const float *params, void *packed, hipStream_t st) {
  hipLaunchKernelGGL(k_mlp_pack, dim3((kPAll + 255) / 256), dim3(256), 0, st, params, static_cast<bf16x8 *>(packed));
  return hipGetLastError();
}

}  // namespace dh

using namespace dh;

namespace {
thread_local std::string g_mlp_err;
int mlp_fail(int code, const std::string &msg) {
  g_mlp_err = msg;
  return code;
}
// blocks of k_mlp_train: one per 64-sample tile up to two per CU (57 KB of
// LDS each); more samples loop
constexpr long long kTrBlocks = 512;
long long train_blocks(long long n) { return std::min<long long>(kTrBlocks, (n + kTrTile - 1) / kTrTile); }
}  // namespace

extern "C" {

const char *dh_mlp_last_error(void) { return g_mlp_err.c_str(); }

int32_t dh_mlp_nparams(void) { return kMlpNP; }

int64_t dh_mlp_packed_bytes(void) { return 16LL * kPAll; }

int64_t dh_mlp_work_bytes(int64_t n) {
  if (n <= 0) return 0;
  return 4LL * train_blocks(n) * kPartLd;
}

int dh_mlp_pack_dev(const float *params, void *packed, void *stream) {
  if (!params || !packed) return mlp_fail(DH_EARG, "null pointer");
  hipLaunchKernelGGL(k_mlp_pack, dim3((kPAll + 255) / 256), dim3(256), 0, static_cast<hipStream_t>(stream), params,
                     static_cast<bf16x8 *>(packed));
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? DH_OK : mlp_fail(DH_EHIP, hipGetErrorString(e));
}

int dh_mlp_infer_dev(const void *packed, const float *params, const float *x, int64_t ld, int64_t n, float scale,
                     float *out, void *stream) {
  if (!packed || !params || !x || !out) return mlp_fail(DH_EARG, "null pointer");
  if (n <= 0 || ld < n) return mlp_fail(DH_EARG, "need 0 < n <= ld");
  if (ld > (1LL << 27)) return mlp_fail(DH_EARG, "ld must be below 2^27");
  const long long waves = std::min<long long>((n + 15) / 16, 4096);
  hipLaunchKernelGGL(k_mlp_infer, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const bf16x8 *>(packed), params, x, (long long)ld, (long long)n, scale, out);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? DH_OK : mlp_fail(DH_EHIP, hipGetErrorString(e));
}

int dh_mlp_grad_dev(const float *params, const void *packed, const float *x, const float *target, int64_t n,
                    void *work, int64_t work_bytes, float *grad, float *loss, void *stream) {
  if (!params || !packed || !x || !target || !work || !grad || !loss) return mlp_fail(DH_EARG, "null pointer");
  if (n <= 0 || n % 32 != 0) return mlp_fail(DH_EARG, "the batch must be a positive multiple of 32 samples");
  if (n > (1LL << 24)) return mlp_fail(DH_EARG, "the batch must hold at most 2^24 samples");
  if (work_bytes < dh_mlp_work_bytes(n)) return mlp_fail(DH_EARG, "work buffer smaller than dh_mlp_work_bytes(n)");
  hipStream_t st = static_cast<hipStream_t>(stream);
  float *part = static_cast<float *>(work);
  const int nb = (int)train_blocks(n);
  hipLaunchKernelGGL(k_mlp_train, dim3(nb), dim3(kTrThreads), 0, st, static_cast<const bf16x8 *>(packed), params, x,
                     target, (long long)n, 1.0f / (float)n, part);
  hipLaunchKernelGGL(k_mlp_reduce, dim3((kMlpNP + 1 + 63) / 64), dim3(256), 0, st, part, nb, grad, loss);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? DH_OK : mlp_fail(DH_EHIP, hipGetErrorString(e));
}

int dh_mlp_adam_dev(float *params, float *m, float *v, const float *grad, float lr, int32_t step, void *packed,
                    void *stream) {
  if (!params || !m || !v || !grad || !packed) return mlp_fail(DH_EARG, "null pointer");
  if (step < 1) return mlp_fail(DH_EARG, "Adam steps count from 1");
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(k_mlp_adam_pack, dim3((kMlpNP + 63) / 64), dim3(64), 0, st, params, m, v, grad, lr, b1, b2, 1e-8f,
                     c1, c2, static_cast<bf16x8 *>(packed));
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? DH_OK : mlp_fail(DH_EHIP, hipGetErrorString(e));
}

}  // extern "C"
