// Training and evaluation kernels of the surrogate network (layout: mlp.hpp).
//
// One training step over a minibatch of B samples (B a multiple of 256), two launches:
//   k_train   one wavefront per 16 samples, 8 wavefronts per block: standardise, forward
//             (MFMA), loss gradient, backward to the pre-activation gradients (MFMA with the
//             transposed weights); the network and the bf16 activations and gradients of the
//             block's 128 samples are in LDS, the latter feature-major, and the block sums its
//             weight gradients dW = dZ^T H from there (MFMA, the samples are the k dimension);
//             FP32 partials per block
//   k_adam    sums the partials (in FP64), applies Adam to the FP32 master parameters and
//             refreshes the bf16 operand copies of each weight
// The loss is the mean over samples and the 8 outputs of (y - (t - mu_out) / sig_out)^2.
#include <hip/hip_runtime.h>

#include <cstddef>

#include "mlp_device.hpp"
#include "mlp_kernels.hpp"

namespace ppk {
namespace mlpk {

using namespace mlpd;

constexpr int kWaveSamples = 64;  // inference: samples per wavefront
constexpr int kTrainWaves = 8, kGroup = 16 * kTrainWaves;  // k_train: samples per pass of a block
constexpr int kMaxTrainBlocks = 256;  // the CUs of an MI355X, on any device, so that the order of
                                      // the sums is the same; more groups are walked with this stride
constexpr int kAdamParts = 4;  // k_adam: most threads per parameter
// row stride of the feature-major LDS arrays: 8 samples more than a group, so that the 16 rows
// of an operand load start 4 banks apart
constexpr int kSP = kGroup + 8;

// sample index of minibatch slot i of training step `step` (uniform with replacement)
__device__ __forceinline__ long long pick(unsigned long long seed, long long step, long long i,
                                          long long n) {
  unsigned long long z = seed + 0x9E3779B97F4A7C15ull * (unsigned long long)(step * 0x10001 + i + 1);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return (long long)(z % (unsigned long long)n);
}

// standardised bf16 features of the wave's samples into sX, raw targets into sT
__device__ __forceinline__ void stage_samples(const MlpView &w, const float *X, const float *T,
                                              long long idx, uint16_t *sX, float *sT) {
  const int lane = lane_id();
  const float *x = X + idx * kMlpIn;
#pragma unroll
  for (int i = 0; i < kMlpIn; ++i) sX[lane * 16 + i] = bf16_bits((x[i] - w.mu_in[i]) * w.isig_in[i]);
  if (T) {
    const float *t = T + idx * kMlpOut;
#pragma unroll
    for (int o = 0; o < kMlpOut; ++o) sT[lane * 8 + o] = (t[o] - w.mu_out[o]) / w.sig_out[o];
  }
}

// LDS of a training block.  The operand copies of the network lie over arrays that a group writes
// later: the forward ones over H2 and Z2, the transposed W2 with the biases over Z1.
struct TrainLds {
  uint16_t H1[128 * kSP], H2[128 * kSP], Z2[128 * kSP], Z1[128 * kSP];  // activations, gradients
  uint16_t XT[16 * kSP], DY[16 * kSP];  // features, output gradients (rows 8..15 zero)
  uint16_t X[kTrainWaves][16 * 16];     // features, sample-major
  float T[kTrainWaves][16 * 8];         // standardised targets
};
static_assert(sizeof(TrainLds) <= 160 * 1024, "training block exceeds the LDS of a CU");
constexpr int kNetAt = (int)(offsetof(TrainLds, Z1) - offsetof(MlpPacked, A2T));
static_assert(kNetAt % 16 == 0 && kNetAt >= (int)offsetof(TrainLds, H2) &&
                  kNetAt + sizeof(MlpPacked) <= offsetof(TrainLds, XT) &&
                  sizeof(MlpPacked) % 16 == 0,
              "the network does not lie over H2, Z2 and Z1");

// Rows r and r + 1 of a feature-major array from the bf16 pair (r, r + 1) that each lane holds for
// its sample: neighbouring lanes swap, so that the even one writes row r and the odd one row r + 1,
// two samples each (half the writes of one value per lane).
__device__ __forceinline__ void put_pair(uint16_t *A, int r, int sc, unsigned mine) {
  const unsigned other = (unsigned)__builtin_amdgcn_mov_dpp((int)mine, 0xB1, 0xf, 0xf, true);
  const bool odd = sc & 1;
  const unsigned v = odd ? (other >> 16) | (mine & 0xffff0000u) : (mine & 0xffffu) | (other << 16);
  *reinterpret_cast<unsigned *>(A + (r + (odd ? 1 : 0)) * kSP + (sc & ~1)) = v;
}
__device__ __forceinline__ void put_rows(uint16_t *A, int sc, int g, const v8bf (&b)[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const v4u w = __builtin_bit_cast(v4u, b[q]);
#pragma unroll
    for (int p = 0; p < 4; ++p) put_pair(A, mlp_feat(q, g, 2 * p), sc, w[p]);
  }
}
// operand of a 16x16x32 step over samples: lane l holds 8 samples from 8 (l / 16) of row l % 16
__device__ __forceinline__ v8bf ld_rows(const uint16_t *A, int row, int k) {
  const int lane = lane_id();
  return *reinterpret_cast<const v8bf *>(A + (row + (lane & 15)) * kSP + k + 8 * (lane >> 4));
}
// A minibatch of 4096 is 32 blocks of 8 wavefronts.  The time is one group's chain of loads and
// MFMAs, not work (0.5 GFLOP a step), so a wavefront takes 16 samples only (64 per wavefront and
// the activations in memory between two kernels: 117 us a step).  k_adam has just rewritten the
// network, so its first reads miss every cache: the block fetches it whole into LDS with all loads
// in flight, where each wavefront reading its operands as it came to them met those misses one
// after another and moved 64 KB through the L1 cache (a step 31 us, now 18.6: k_train 14, k_adam
// 4.6; over 262144 samples, 8 groups per block, 134 us, now 92).
__global__ void __launch_bounds__(64 * kTrainWaves)
k_train(const MlpPacked *__restrict__ net, const float *__restrict__ X,
        const float *__restrict__ T, const long long *idx, long long n, unsigned long long seed,
        long long step, long long B, float *partials, float inv_count) {
  __shared__ __attribute__((aligned(16))) TrainLds S;
  const MlpPacked *img = reinterpret_cast<const MlpPacked *>(reinterpret_cast<char *>(&S) + kNetAt);
  const MlpView w = view_of(img);
  const int wave = threadIdx.x >> 6, lane = lane_id(), g = lane >> 4, col = lane & 15;
  uint16_t *sX = S.X[wave];
  float *sT = S.T[wave];
  const int sc = 16 * wave + col;  // this lane's sample column in the feature-major arrays
  for (int k = threadIdx.x; k < 8 * kSP; k += 64 * kTrainWaves) S.DY[8 * kSP + k] = 0;
  // gradients of this wavefront: dW2 tiles (a, wave), then dW1 tile wave, dW3 tile wave, and the
  // sums of rows 16 wave of Z1 and Z2 and of DY (products with ones)
  v4f acc[13];
#pragma unroll
  for (int a = 0; a < 13; ++a) acc[a] = v4f{0.f, 0.f, 0.f, 0.f};

#pragma unroll 1
  for (long long grp = blockIdx.x; grp < B / kGroup; grp += gridDim.x) {
    {  // the network and the samples, all loads in flight at once
      constexpr int kChunks = sizeof(MlpPacked) / 16, kThreads = 64 * kTrainWaves;
      constexpr int kPer = (kChunks + kThreads - 1) / kThreads;
      const uint4 *src = reinterpret_cast<const uint4 *>(net);
      uint4 c[kPer];
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const int i = k * kThreads + threadIdx.x;
        c[k] = src[i < kChunks ? i : kChunks - 1];
      }
      // four lanes per sample: four features and two targets each
      const int s = lane >> 2, part = lane & 3;
      const long long slot = grp * kGroup + 16 * wave + s;
      const long long sample = idx ? idx[slot] : pick(seed, step, slot, n);
      const float4 x = *reinterpret_cast<const float4 *>(X + sample * kMlpIn + 4 * part);
      const float2 t = *reinterpret_cast<const float2 *>(T + sample * kMlpOut + 2 * part);
      uint4 *dst = reinterpret_cast<uint4 *>(reinterpret_cast<char *>(&S) + kNetAt);
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const int i = k * kThreads + threadIdx.x;
        if (i < kChunks) dst[i] = c[k];
      }
      __syncthreads();
      const float xv[4] = {x.x, x.y, x.z, x.w}, tv[2] = {t.x, t.y};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * part + e;
        const uint16_t v = bf16_bits((xv[e] - w.mu_in[i]) * w.isig_in[i]);
        sX[s * 16 + i] = v;
        S.XT[i * kSP + 16 * wave + s] = v;
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int o = 2 * part + e;
        sT[s * 8 + o] = (tv[e] - w.mu_out[o]) / w.sig_out[o];
      }
    }
    wave_lds_sync();
    const v4s xb = *reinterpret_cast<const v4s *>(sX + col * 16 + 4 * g);
    v8bf h1b[4], h2b[4];
    unsigned m1, m2;
    v4f y;
    mlp_forward16(w, xb, h1b, h2b, m1, m2, y);
    v4s a3t[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) a3t[r] = ld_a16(w.A3T, r, lane);
    __syncthreads();  // H2 and Z2 take the place of the forward operands
    // the bf16 activations as the forward pass used them (element e of pair q: feature
    // feat(q, g, e))
    put_rows(S.H1, sc, g, h1b);
    put_rows(S.H2, sc, g, h2b);
    // loss gradient (outputs 4g + j of sample col)
    float dy[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      dy[j] = g < 2 ? 2.f * (y[j] - sT[col * 8 + ((4 * g + j) & 7)]) * inv_count : 0.f;
    const unsigned dyw[2] = {bf16x2(dy[0], dy[1]), bf16x2(dy[2], dy[3])};
    const v4s dyb = __builtin_bit_cast(v4s, dyw);
    if (g < 2) {
      put_pair(S.DY, 4 * g, sc, dyw[0]);
      put_pair(S.DY, 4 * g + 2, sc, dyw[1]);
    }
    // dH2 = W3^T dY, dZ2 = dH2 * (z2 > 0), packed in pairs as the B operands of dH1
    v8bf db[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      v4f t[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int r = 2 * q + h;
        const v4f c = mfma_k16(a3t[r], dyb, v4f{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int j = 0; j < 4; ++j) t[h][j] = (m2 >> (4 * r + j)) & 1u ? c[j] : 0.f;
      }
      db[q] = pack_pair(t[0], t[1]);
    }
    put_rows(S.Z2, sc, g, db);
    // dH1 = W2^T dZ2, dZ1 = dH1 * (z1 > 0)
    v8bf da[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      v4f t[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int r = 2 * p + h;
        v4f c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 4; ++q) c = mfma_k32(ld_a32(w.A2T, r * 4 + q, lane), db[q], c);
#pragma unroll
        for (int j = 0; j < 4; ++j) t[h][j] = (m1 >> (4 * r + j)) & 1u ? c[j] : 0.f;
      }
      da[p] = pack_pair(t[0], t[1]);
    }
    __syncthreads();  // Z1 takes the place of the transposed W2
    put_rows(S.Z1, sc, g, da);
    __syncthreads();
    // gradients over the group's samples
    const __bf16 one = (__bf16)1.f;
    const v8bf ones = {one, one, one, one, one, one, one, one};
#pragma unroll
    for (int k = 0; k < kGroup; k += 32) {
      const v8bf h1 = ld_rows(S.H1, 16 * wave, k);
#pragma unroll
      for (int a = 0; a < 8; ++a) acc[a] = mfma_k32(ld_rows(S.Z2, 16 * a, k), h1, acc[a]);
      const v8bf z1 = ld_rows(S.Z1, 16 * wave, k), dyr = ld_rows(S.DY, 0, k);
      acc[8] = mfma_k32(z1, ld_rows(S.XT, 0, k), acc[8]);
      acc[9] = mfma_k32(dyr, ld_rows(S.H2, 16 * wave, k), acc[9]);
      acc[10] = mfma_k32(z1, ones, acc[10]);
      acc[11] = mfma_k32(ld_rows(S.Z2, 16 * wave, k), ones, acc[11]);
      acc[12] = mfma_k32(dyr, ones, acc[12]);
    }
    __syncthreads();
  }

  float *P = partials + (long long)blockIdx.x * kMlpTrained;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = 4 * g + j;
#pragma unroll
    for (int a = 0; a < 8; ++a) P[kMlpW2 + (16 * a + i) * 128 + 16 * wave + col] = acc[a][j];
    P[kMlpW1 + (16 * wave + i) * 16 + col] = acc[8][j];
    if (i < 8) P[kMlpW3 + i * 128 + 16 * wave + col] = acc[9][j];
    if (col == 0) {
      P[kMlpB1 + 16 * wave + i] = acc[10][j];
      P[kMlpB2 + 16 * wave + i] = acc[11][j];
      if (wave == 0 && i < 8) P[kMlpB3 + i] = acc[12][j];
    }
  }
}

// the packed copies of trained parameter i (the inverse of pack_weight)
__device__ __forceinline__ void repack(MlpPacked *net, int i, float p) {
  const uint16_t v = bf16_bits(p);
  auto feat = [](int f, int &q, int &g, int &e) {  // inverse of mlp_feat
    q = f >> 5;
    const int r = f & 31;
    g = (r & 15) >> 2;
    e = (r & 3) + (r < 16 ? 0 : 4);
  };
  int q, g, e;
  if (i < kMlpB1) {
    const int o = i >> 4, c = i & 15;
    net->A1[o >> 4][(c >> 2) * 16 + (o & 15)][c & 3] = v;
  } else if (i < kMlpW2) {
    net->b1[i - kMlpB1] = p;
  } else if (i < kMlpB2) {
    const int o = (i - kMlpW2) >> 7, f = (i - kMlpW2) & 127;
    feat(f, q, g, e);
    net->A2[o >> 4][q][g * 16 + (o & 15)][e] = v;
    feat(o, q, g, e);
    net->A2T[f >> 4][q][g * 16 + (f & 15)][e] = v;
  } else if (i < kMlpW3) {
    net->b2[i - kMlpB2] = p;
  } else if (i < kMlpB3) {
    const int o = (i - kMlpW3) >> 7, f = (i - kMlpW3) & 127;
    feat(f, q, g, e);
    net->A3[q][g * 16 + o][e] = v;
    net->A3T[f >> 4][(o >> 2) * 16 + (f & 15)][o & 3] = v;
  } else {
    net->b3[i - kMlpB3] = p;
  }
}

// blockDim.x / 64 threads per parameter (adam_parts), which share its partials
__global__ void __launch_bounds__(64 * kAdamParts)
k_adam(const float *__restrict__ partials, int nparts, float *P, float *m, float *v,
       float *grad_out, MlpPacked *net, int step, float lr, float beta1, float beta2, float eps) {
  __shared__ double part[kAdamParts][64];
  const int lane = lane_id(), w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int i = blockIdx.x * 64 + lane;
  double sum = 0.0;
  if (i < kMlpTrained) {
#pragma unroll 16
    for (int c = w; c < nparts; c += nw) sum += partials[(long long)c * kMlpTrained + i];
  }
  if (nw > 1) {
    part[w][lane] = sum;
    __syncthreads();
    if (w > 0) return;
    for (int c = 1; c < nw; ++c) sum += part[c][lane];
  }
  if (i >= kMlpTrained) return;
  const float gsum = (float)sum;
  if (grad_out) grad_out[i] = gsum;
  if (lr == 0.f) return;  // gradient only
  const float mi = beta1 * m[i] + (1.f - beta1) * gsum;
  const float vi = beta2 * v[i] + (1.f - beta2) * gsum * gsum;
  m[i] = mi;
  v[i] = vi;
  const float mh = mi / (1.f - __powf(beta1, (float)step));
  const float vh = vi / (1.f - __powf(beta2, (float)step));
  const float p = P[i] - lr * mh / (sqrtf(vh) + eps);
  P[i] = p;
  repack(net, i, p);
}

__global__ void k_pack(const float *P, MlpPacked *net) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  uint16_t *W = &net->A1[0][0][0];
  if (n < kPackWeights) W[n] = pack_weight(P, n);
  if (n < 128) {
    net->b1[n] = P[kMlpB1 + n];
    net->b2[n] = P[kMlpB2 + n];
  }
  if (n < 16) {
    net->b3[n] = n < 8 ? P[kMlpB3 + n] : 0.f;
    net->mu_in[n] = P[kMlpMuIn + n];
    net->isig_in[n] = P[kMlpIsigIn + n];
  }
  if (n < 8) {
    net->mu_out[n] = P[kMlpMuOut + n];
    net->sig_out[n] = P[kMlpSigOut + n];
  }
}

// inference on n samples (features X[n][16]) -> Y[n][8] (standardised outputs) and, with
// targets, per-block partial sums of squared errors per output
__global__ void __launch_bounds__(256) k_infer(const MlpPacked *__restrict__ net,
                                               const float *__restrict__ X,
                                               const float *__restrict__ T, long long n,
                                               float *Y, double *sq_parts) {
  __shared__ __attribute__((aligned(16))) uint16_t sXall[4][64 * 16];
  __shared__ float sTall[4][64 * 8];
  __shared__ float sYall[4][64 * 8];
  __shared__ double red[256];
  const MlpView w = view_of(net);
  const int wave = threadIdx.x >> 6, lane = lane_id();
  const long long me = ((long long)blockIdx.x * 4 + wave) * kWaveSamples + lane;
  uint16_t *sX = sXall[wave];
  float *sT = sTall[wave], *sY = sYall[wave];
  stage_samples(w, X, T, me < n ? me : n - 1, sX, sT);
  wave_lds_sync();
  mlp_infer_wave(w, sX, sY);
  double sq[8];
#pragma unroll
  for (int o = 0; o < 8; ++o) {
    const float y = sY[lane * 8 + o];
    if (me < n && Y) Y[me * 8 + o] = y;
    const double d = T && me < n ? (double)y - (double)sT[lane * 8 + o] : 0.0;
    sq[o] = d * d;
  }
  if (!sq_parts) return;
#pragma unroll 1
  for (int o = 0; o < 8; ++o) {
    red[threadIdx.x] = sq[o];
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
      if (threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
      __syncthreads();
    }
    if (threadIdx.x == 0) sq_parts[(long long)blockIdx.x * 8 + o] = red[0];
    __syncthreads();
  }
}

// per-block sums and sums of squares of the 16 features and 8 targets (standardisation)
__global__ void __launch_bounds__(256) k_moments(const float *__restrict__ X,
                                                 const float *__restrict__ T, long long n,
                                                 double *parts) {
  __shared__ double red[256];
  const long long per = (n + gridDim.x - 1) / gridDim.x;
  const long long lo = (long long)blockIdx.x * per, hi = lo + per < n ? lo + per : n;
#pragma unroll 1
  for (int c = 0; c < 24; ++c) {
    double s = 0.0, s2 = 0.0;
    for (long long i = lo + threadIdx.x; i < hi; i += 256) {
      const double v = c < 16 ? X[i * 16 + c] : T[i * 8 + c - 16];
      s += v;
      s2 += v * v;
    }
    for (int k = 0; k < 2; ++k) {
      red[threadIdx.x] = k ? s2 : s;
      __syncthreads();
      for (int st = 128; st > 0; st >>= 1) {
        if (threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
        __syncthreads();
      }
      if (threadIdx.x == 0) parts[((long long)blockIdx.x * 24 + c) * 2 + k] = red[0];
      __syncthreads();
    }
  }
}

}  // namespace mlpk

// ---- launchers (mlp_kernels.hpp) -----------------------------------------------------------
namespace mlp {

int train_blocks(long long B) {
  const long long g = B / mlpk::kGroup;
  return (int)(g < mlpk::kMaxTrainBlocks ? g : mlpk::kMaxTrainBlocks);
}

// One thread per parameter sums the 32 partials of a 4096 minibatch in two rounds of 16 loads, and
// more wavefronts only cost their start (a step 18.6 us, with four threads 19.9); 256 partials are
// 16 rounds, or four with four threads (a step over 32768 samples 32.7 us, now 28.7).
static int adam_parts(int nparts) { return nparts > 64 ? mlpk::kAdamParts : 1; }

hipError_t train_step(MlpPacked *net, float *P, float *m, float *v, const float *X,
                      const float *T, const long long *idx, long long n, unsigned long long seed,
                      long long step, long long B, float *partials, float *grad_out, float lr,
                      hipStream_t s) {
  using namespace mlpk;
  if (B < kGroup || B % kGroup) return hipErrorInvalidValue;
  const float inv_count = 1.f / (float)(B * kMlpOut);
  const int nb = train_blocks(B);
  hipLaunchKernelGGL(k_train, dim3((unsigned)nb), dim3(64 * kTrainWaves), 0, s, net, X, T,
                     idx, n, seed, step, B, partials, inv_count);
  hipLaunchKernelGGL(k_adam, dim3((kMlpTrained + 63) / 64), dim3(64 * adam_parts(nb)), 0, s, partials, nb, P, m, v,
                     grad_out, net, (int)(step + 1), lr, 0.9f, 0.999f, 1e-8f);
  return hipGetLastError();
}

hipError_t pack(const float *P, MlpPacked *net, hipStream_t s) {
  hipLaunchKernelGGL(mlpk::k_pack, dim3((kPackWeights + 255) / 256), dim3(256), 0, s, P, net);
  return hipGetLastError();
}

int infer_blocks(long long n) { return (int)((n + 255) / 256); }

hipError_t infer(const MlpPacked *net, const float *X, const float *T, long long n, float *Y,
                 double *sq_parts, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(mlpk::k_infer, dim3((unsigned)infer_blocks(n)), dim3(256), 0, s, net, X, T,
                     n, Y, sq_parts);
  return hipGetLastError();
}

hipError_t moments(const float *X, const float *T, long long n, double *parts, int nblocks,
                   hipStream_t s) {
  hipLaunchKernelGGL(mlpk::k_moments, dim3(nblocks), dim3(256), 0, s, X, T, n, parts);
  return hipGetLastError();
}

}  // namespace mlp
}  // namespace ppk
