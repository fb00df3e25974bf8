// mlp.hip -- see mlp.h.
//
// A training step is three launches on bf16 MFMA with fp32 accumulation:
// BatchKernel (forward, loss and the gradient down to the embeddings, 16 rows
// of the batch per block), WeightGradKernel (what contracts over the batch)
// and AdamKernel.  Sums over blocks go through stored partial sums: float
// atomics of blocks on different XCDs meet in memory, 10 ns each on one
// address.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <vector>

#include "cost_model.h"
#include "cost_model_gpu.h"
#include "gz_runtime.h"
#include "gz_common.h"
#include "gz_device.h"
#include "mlp.h"

namespace gz {

namespace {

typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));

constexpr size_t kOffEmbed = 0;
constexpr size_t kOffW1 = kOffEmbed + (size_t)kCostAlphabet * kCostEmbed;
constexpr size_t kOffB1 = kOffW1 + (size_t)kCostH1 * kCostIn;
constexpr size_t kOffW2 = kOffB1 + kCostH1;
constexpr size_t kOffB2 = kOffW2 + (size_t)kCostH2 * kCostH1;
constexpr size_t kOffW3 = kOffB2 + kCostH2;
constexpr size_t kOffB3 = kOffW3 + kCostH2;
constexpr size_t kFlat = kOffB3 + 1;

__device__ __forceinline__ uint16_t F2Bf(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float Bf2F(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ float Gelu(float z) {
  return 0.5f * z * (1.f + erff(z * 0.70710678118654752f));
}
__device__ __forceinline__ float GeluGrad(float z) {
  const float cdf = 0.5f * (1.f + erff(z * 0.70710678118654752f));
  const float pdf = 0.39894228040143268f * expf(-0.5f * z * z);
  return cdf + z * pdf;
}

typedef __bf16 gemm_bf16x8 __attribute__((ext_vector_type(8)));
typedef float gemm_float4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// Training, first kernel: a block of four waves takes 16 rows of the batch
// from their codes to the embedding gradient; layer inputs, pre-activations
// and dX stay in registers and LDS.
//
// Tiles are v_mfma_f32_16x16x32_bf16: lane l supplies A[row l % 16][k] and
// B[k][column l % 16] for k = 8 (l / 16) + j, j < 8; accumulator register r
// holds C[4 (l / 16) + r][l % 16].  A wave owns 64 of the first layer's 256
// units (four tiles), 16 of the second's 64, 256 of the 1024 inputs.  The
// weights are kept once more in the order in which the lanes read them (a
// tile's operand is 1 KB in a row; of the row-major weights it is 16 pieces
// 2 KB apart) and
// go from L2 straight into B operands, 16 of them ahead.  A operands of layer 1
// are one residue's embedding each (kCostEmbed = 8), read by code from LDS.
// Bound: a block's serial phases (one block per CU at 4,096 rows) and their
// instruction fetches: a launch runs each line once or a few times, so that
// loops unrolled into 40 KB of code took 77 us where these 10 KB take 41.
// At 4,096 rows the work of this kernel took 160 us as 13 launches (embedding,
// layers, output, loss, column sums, dZ2, dZ1, dX, embedding gradient).
// ---------------------------------------------------------------------------
constexpr int kRows = 16;        // of the batch per block
constexpr int kTileK = 32;       // of one MFMA
constexpr int kGroup = 4;        // k steps read together
constexpr int kGroups = kCostIn / (kTileK * kGroup);
constexpr int kWaveUnits = kCostH1 / 4;
constexpr int kWaveTiles = kWaveUnits / 16;
constexpr int kInputTiles = kCostIn / 4 / 16;  // of a wave
constexpr int kH1Steps = kCostH1 / kTileK, kH2Steps = kCostH2 / kTileK;

// Where operand value (column n, k) of a product over K values is kept.
__device__ __forceinline__ size_t OperandAt(int n, int k, int K) {
  return (size_t)(n / 16 * (K / kTileK) + k / kTileK) * (16 * kTileK) +
         (n % 16 + k % kTileK / 8 * 16) * 8 + k % 8;
}
// This lane's part of the operand of columns 16 tile .. + 16, k step `step`.
__device__ __forceinline__ gemm_bf16x8 Operand(const uint16_t *p, int tile, int step, int K) {
  return *reinterpret_cast<const gemm_bf16x8 *>(
      p + (size_t)(tile * (K / kTileK) + step) * (16 * kTileK) + (threadIdx.x & 63) * 8);
}

// The weights in operand order: W1 by unit (k: inputs) and by input (k:
// units), W2 by unit and by hidden unit.
struct Operands {
  uint16_t *w1, *w1t, *w2, *w2t;
};

static_assert(kOffW3 == kOffB2 + kCostH2 && kOffB3 == kOffW3 + kCostH2, "sums in weight order");
static_assert(kCostEmbed == 8 && kCostH1 == 256 && kCostH2 == 64, "the block's tiles");

// The batch's rows: row r < n is row order[r] (r without order) of codes and
// targets; rows past n read code 20 and count nothing.
struct BatchRows {
  const uint8_t *codes;
  const float *targets;
  const uint32_t *order;
  int n;
};

// A block's sums over its rows: the gradients of the embedding, of the biases
// and of the output weights, and the loss.
constexpr int kSumB1 = kCostAlphabet * kCostEmbed, kSumB2 = kSumB1 + kCostH1,
              kSumW3 = kSumB2 + kCostH2, kSumB3 = kSumW3 + kCostH2, kSumLoss = kSumB3 + 1,
              kSums = kSumLoss + 1;
constexpr int kMostBatchBlocks = 1024;

__global__ void __launch_bounds__(256, 1)
    BatchKernel(BatchRows rows, int tiles, const uint16_t *embh, Operands weights,
                const float *b1, const float *b2, const float *w3, const float *b3,
                uint8_t *batch_codes, uint16_t *h1, uint16_t *dz2h, uint16_t *dz1h, float *sums) {
  constexpr int kPad = 8;
  __shared__ uint4 emb[kCostAlphabet];
  __shared__ __align__(16) uint32_t codes[kRows][kCostResidues / 4 + 1];
  __shared__ __align__(16) uint16_t tile[kRows][kCostH1 + kPad];  // h1, then dz1
  __shared__ __align__(16) uint16_t dz2t[kRows][kCostH2 + kPad];
  __shared__ float z1t[kRows][kCostH1 + 4], dh1t[kRows][kCostH1 + 4];
  __shared__ float zt[kRows][kCostH2 + 1], pt[kRows][kCostH2 + 1];
  __shared__ float w3s[kCostH2];
  __shared__ float part[2][4];
  __shared__ float table[kCostAlphabet * kCostEmbed];
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const int l16 = lane & 15, quarter = lane >> 4;
  const int hr = t >> 4;  // the row of 16 threads
  const float bias1 = b1[t], bias2 = b2[wave * 16 + l16], bias3 = b3[0];
  if (t < kCostAlphabet) emb[t] = reinterpret_cast<const uint4 *>(embh)[t];
  if (t < kCostAlphabet * kCostEmbed) table[t] = 0.f;
  if (t < kCostH2) w3s[t] = Bf2F(F2Bf(w3[t]));
  float sum1 = 0.f, sum2 = 0.f;  // of unit t's dZ1, and of what thread t sums below
  for (int row_tile = blockIdx.x; row_tile < tiles; row_tile += gridDim.x) {
    const int base = row_tile * kRows;
    // layer 1's weights: group g's operand of k step s and tile i
    gemm_bf16x8 w[2][kGroup][kWaveTiles];
    auto read_group = [&](int g, gemm_bf16x8 (&v)[kGroup][kWaveTiles]) {
#pragma unroll
      for (int i = 0; i < kWaveTiles; ++i)
#pragma unroll
        for (int s = 0; s < kGroup; ++s)
          v[s][i] = Operand(weights.w1, wave * kWaveTiles + i, g * kGroup + s, kCostIn);
    };
    // the rows' codes, 16 threads of eight each
    float target = 0.f;
    {
      const int b = base + hr, k = (t & 15) * 2;
      uint2 c = make_uint2(0x14141414u, 0x14141414u);
      if (b < rows.n) {
        const size_t at = rows.order ? rows.order[b] : (uint32_t)b;
        c = *reinterpret_cast<const uint2 *>(rows.codes + at * kCostResidues + k * 4);
        target = rows.targets[at];
      }
      codes[hr][k] = c.x;
      codes[hr][k + 1] = c.y;
      *reinterpret_cast<uint2 *>(batch_codes + (size_t)b * kCostResidues + k * 4) = c;
    }
    read_group(0, w[0]);
    __syncthreads();
    gemm_float4 acc[kWaveTiles];
#pragma unroll
    for (int i = 0; i < kWaveTiles; ++i) acc[i] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int g0 = 0; g0 < kGroups; g0 += 2) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int g = g0 + h;
        read_group(g + 1 < kGroups ? g + 1 : g, w[h ^ 1]);  // (the last one again)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < kGroup; ++s) {
          // residue 4 (g kGroup + s) + quarter of the lane's row
          const uint32_t c = (codes[l16][g * kGroup + s] >> (8 * quarter)) & 0xffu;
          const gemm_bf16x8 a = *reinterpret_cast<const gemm_bf16x8 *>(
              &emb[c < (uint32_t)kCostAlphabet ? c : kCostAlphabet - 1]);
#pragma unroll
          for (int i = 0; i < kWaveTiles; ++i)
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w[h][s][i], acc[i], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // the second layer's operands, in flight during the GELUs
    gemm_bf16x8 v2[kH1Steps], vt[kH2Steps][kWaveTiles];
#pragma unroll
    for (int s = 0; s < kH1Steps; ++s) v2[s] = Operand(weights.w2, wave, s, kCostH1);
#pragma unroll
    for (int s = 0; s < kH2Steps; ++s)
#pragma unroll
      for (int i = 0; i < kWaveTiles; ++i)
        vt[s][i] = Operand(weights.w2t, wave * kWaveTiles + i, s, kCostH2);
#pragma unroll
    for (int i = 0; i < kWaveTiles; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        z1t[4 * quarter + r][wave * kWaveUnits + i * 16 + l16] = acc[i][r];
    __syncthreads();
    // z1 and h1, a unit per thread
#pragma unroll 2
    for (int r = 0; r < kRows; ++r) {
      const float z = z1t[r][t] + bias1;
      z1t[r][t] = z;
      tile[r][t] = F2Bf(Gelu(z));
    }
    __syncthreads();
    auto store_tile = [&](uint16_t *out) {  // 16 threads per row, 16 values each
      const int c = (t & 15) * 16;
      uint4 *o = reinterpret_cast<uint4 *>(out + (size_t)(base + hr) * kCostH1 + c);
      const uint4 *x = reinterpret_cast<const uint4 *>(&tile[hr][c]);
      o[0] = x[0];
      o[1] = x[1];
    };
    store_tile(h1);
    {
      gemm_float4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < kH1Steps; ++s)
        z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *reinterpret_cast<const gemm_bf16x8 *>(&tile[l16][s * kTileK + 8 * quarter]), v2[s],
            z, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) zt[4 * quarter + r][wave * 16 + l16] = z[r] + bias2;
    }
    __syncthreads();
    // the head, 16 threads per row and four units each: output, mean squared
    // error and its gradient, dZ2 = dY w3 * gelu'(Z2)
    {
      const int c0 = (t & 15) * 4, b = base + hr;
      float s = 0.f;
#pragma unroll 1
      for (int c = c0; c < c0 + 4; ++c) {
        const float h = Bf2F(F2Bf(Gelu(zt[hr][c])));
        pt[hr][c] = h;
        s += h * w3s[c];
      }
#pragma unroll
      for (int m = 1; m < 16; m <<= 1) s += __shfl_xor(s, m, kWave);
      const float d = b < rows.n ? s + bias3 - target : 0.f;
      const float dy = 2.f * d / rows.n;
#pragma unroll 1
      for (int c = c0; c < c0 + 4; ++c) {
        const float dz = dy * w3s[c] * GeluGrad(zt[hr][c]);
        zt[hr][c] = dz;
        pt[hr][c] *= dy;
        dz2t[hr][c] = F2Bf(dz);
      }
      *reinterpret_cast<uint2 *>(dz2h + (size_t)b * kCostH2 + c0) =
          *reinterpret_cast<const uint2 *>(&dz2t[hr][c0]);
      float e = d * d, g = dy;
      e += __shfl_xor(e, 16, kWave);
      g += __shfl_xor(g, 16, kWave);
      e += __shfl_xor(e, 32, kWave);
      g += __shfl_xor(g, 32, kWave);
      if (lane == 0) {
        part[0][wave] = g;
        part[1][wave] = e;
      }
    }
    __syncthreads();
    // dB2 = sum dZ2, dW3 = H2^T dY, dB3 = sum dY and the loss
    if (t < 2 * kCostH2) {
      const int c = t & (kCostH2 - 1);
      const float(*m)[kCostH2 + 1] = t < kCostH2 ? zt : pt;
#pragma unroll
      for (int r = 0; r < kRows; ++r) sum2 += m[r][c];
    } else if (t < 2 * kCostH2 + 2) {
      const float *p = part[t & 1];
      const float sum = (p[0] + p[1]) + (p[2] + p[3]);
      sum2 += t & 1 ? sum / rows.n : sum;
    }
    // dZ1 = (dZ2 W2) * gelu'(Z1) and dB1 = sum dZ1; the h1 tile is read out
#pragma unroll
    for (int i = 0; i < kWaveTiles; ++i) {
      gemm_float4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < kH2Steps; ++s)
        z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *reinterpret_cast<const gemm_bf16x8 *>(&dz2t[l16][s * kTileK + 8 * quarter]),
            vt[s][i], z, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        dh1t[4 * quarter + r][wave * kWaveUnits + i * 16 + l16] = z[r];
    }
    // dX = dZ1 W1, a wave's 256 inputs two tiles at a time
    constexpr int kPairsOfTiles = kInputTiles / 2;
    gemm_bf16x8 u[2][2][kH1Steps];
    auto read_inputs = [&](int p, gemm_bf16x8 (&v)[2][kH1Steps]) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int s = 0; s < kH1Steps; ++s)
          v[i][s] = Operand(weights.w1t, wave * kInputTiles + 2 * p + i, s, kCostH1);
    };
    read_inputs(0, u[0]);
    __syncthreads();
#pragma unroll 2
    for (int r = 0; r < kRows; ++r) {
      const float dz = dh1t[r][t] * GeluGrad(z1t[r][t]);
      sum1 += dz;
      tile[r][t] = F2Bf(dz);
    }
    __syncthreads();
    store_tile(dz1h);
    gemm_bf16x8 dz[kH1Steps];
#pragma unroll
    for (int s = 0; s < kH1Steps; ++s)
      dz[s] = *reinterpret_cast<const gemm_bf16x8 *>(&tile[l16][s * kTileK + 8 * quarter]);
#pragma unroll 1
    for (int p0 = 0; p0 < kPairsOfTiles; p0 += 2) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int p = p0 + h;
        read_inputs(p + 1 < kPairsOfTiles ? p + 1 : p, u[h ^ 1]);
        __builtin_amdgcn_sched_barrier(0);
        gemm_float4 x[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          x[i] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int s = 0; s < kH1Steps; ++s)
            x[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(dz[s], u[h][i][s], x[i], 0, 0, 0);
        }
        // the embedding gradient: the sum over (row, residue) with code a of
        // the residue's eight columns; a tile is two residues
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int residue = (wave * kInputTiles + 2 * p + i) * 2 + (l16 >> 3);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const uint32_t c =
                (codes[4 * quarter + r][residue >> 2] >> (8 * (residue & 3))) & 0xffu;
            atomicAdd(&table[(c < (uint32_t)kCostAlphabet ? c : kCostAlphabet - 1) * kCostEmbed +
                             (l16 & 7)],
                      x[i][r]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();  // the tile, the codes and the table are read or written
  }
  float *out = sums + (size_t)blockIdx.x * kSums;
  if (t < kCostAlphabet * kCostEmbed) out[t] = table[t];
  out[kSumB1 + t] = sum1;
  if (t < 2 * kCostH2 + 2) out[kSumB2 + t] = sum2;  // dB2, dW3, dB3, the loss
}

// ---------------------------------------------------------------------------
// Training, second kernel: products over 64 x 64 tiles of C[m][n] =
// sum_k A(m, k) B(n, k), a 32 x 32 part per wave (v_mfma_f32_32x32x16_bf16).
// K advances 128 at a time through LDS, where both operand tiles are stored
// k-contiguous; the next two slices are on their way into registers while the
// current one is multiplied.  Sizes are multiples of 64 and rows 16-byte
// aligned.  Values from ke on read 0.
// ---------------------------------------------------------------------------
constexpr int kGemmTile = 64, kGemmK = 128, kGemmPad = 8;
typedef uint16_t GemmLdsTile[kGemmTile][kGemmK + kGemmPad];

// Transposes the k pairs t / 8 + 32 i of rows (t % 8) * 8 .. + 8, v[2 i] the
// even k's values and v[2 i + 1] the odd one's.
__device__ __forceinline__ void StorePairs(GemmLdsTile &T, const uint4 (&v)[4]) {
  const int t = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    uint16_t lo[8], hi[8];
    memcpy(lo, &v[2 * i], 16);
    memcpy(hi, &v[2 * i + 1], 16);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      *reinterpret_cast<uint32_t *>(&T[(t & 7) * 8 + j][2 * ((t >> 3) + 32 * i)]) =
          (uint32_t)lo[j] | (uint32_t)hi[j] << 16;
  }
}

// An operand with unit row stride.
struct ColumnOperand {
  const uint16_t *p;
  long stride;
  struct Slice {
    uint4 v[4];
  };
  __device__ __forceinline__ void Load(Slice &g, int r0, int k0, int ke) const {
    const int t = threadIdx.x;
    const uint16_t *x = p + r0 + (t & 7) * 8;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = k0 + 2 * ((t >> 3) + 32 * (i >> 1)) + (i & 1);
      g.v[i] = k < ke ? *reinterpret_cast<const uint4 *>(x + k * stride) : make_uint4(0, 0, 0, 0);
    }
  }
  __device__ __forceinline__ void Store(GemmLdsTile &T, const Slice &g) const {
    StorePairs(T, g.v);
  }
};

// The batch's embeddings as such an operand: eight rows are one residue.
struct EmbedOperand {
  const uint8_t *codes;
  const uint4 *emb;  // in LDS, zeros behind the alphabet
  struct Slice {
    uint8_t c[4];
  };
  __device__ __forceinline__ void Load(Slice &g, int r0, int k0, int ke) const {
    const int t = threadIdx.x;
    const uint8_t *x = codes + r0 / kCostEmbed + (t & 7);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = k0 + 2 * ((t >> 3) + 32 * (i >> 1)) + (i & 1);
      uint8_t c = kCostAlphabet;
      if (k < ke) {
        c = x[(size_t)k * kCostResidues];
        c = c < kCostAlphabet ? c : (uint8_t)(kCostAlphabet - 1);
      }
      g.c[i] = c;
    }
  }
  __device__ __forceinline__ void Store(GemmLdsTile &T, const Slice &g) const {
    uint4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = emb[g.c[i]];
    StorePairs(T, v);
  }
};

struct GemmLds {
  __align__(16) GemmLdsTile a;
  __align__(16) GemmLdsTile b;
};

// The wave's 32 x 32 part of the tile at (mb, nb) over k [kb, ke).
template <class A, class B>
__device__ __forceinline__ float16_t GemmTile(GemmLds &T, const A &x, const B &y, int mb, int nb,
                                              int kb, int ke) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int am = (wave >> 1) * 32 + (lane & 31), bn = (wave & 1) * 32 + (lane & 31);
  const int kq = (lane >> 5) * 8;
  float16_t acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  typename A::Slice ga[2];
  typename B::Slice gb[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    x.Load(ga[h], mb, kb + h * kGemmK, ke);
    y.Load(gb[h], nb, kb + h * kGemmK, ke);
  }
  for (int k0 = kb; k0 < ke; k0 += 2 * kGemmK) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (k0 + h * kGemmK >= ke) break;
      x.Store(T.a, ga[h]);
      y.Store(T.b, gb[h]);
      __syncthreads();
      x.Load(ga[h], mb, k0 + (h + 2) * kGemmK, ke);
      y.Load(gb[h], nb, k0 + (h + 2) * kGemmK, ke);
#pragma unroll
      for (int ks = 0; ks < kGemmK; ks += 16) {
        const gemm_bf16x8 a = *reinterpret_cast<const gemm_bf16x8 *>(&T.a[am][ks + kq]);
        const gemm_bf16x8 b = *reinterpret_cast<const gemm_bf16x8 *>(&T.b[bn][ks + kq]);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
      }
      __syncthreads();
    }
  }
  return acc;
}

// Row and column inside the tile of accumulator register r of this thread.
__device__ __forceinline__ int TileRow(int r) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  return (wave >> 1) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
}
__device__ __forceinline__ int TileCol() {
  return ((threadIdx.x >> 6) & 1) * 32 + (threadIdx.x & 31);
}

// The batch's slices that the two weight gradients are split into.
struct BatchSplit {
  int w1_slices, w1_rows, w2_slices, w2_rows;  // slices, rows of the batch each
};
constexpr int kW1Tiles = (kCostH1 / kGemmTile) * (kCostIn / kGemmTile);
constexpr int kW2Tiles = kCostH1 / kGemmTile;
constexpr int kMostW1Slices = 8, kMostW2Slices = 32;

// The two weight gradients in one launch: blocks [0, w1) dW1 = dZ1^T X, 64
// tiles times its slices, the others dW2 = dZ2^T H1, 4 tiles times its
// slices, both as partial gradients per slice; then the blocks' sums of the
// first kernel, 64 values a block.  Bound: the latency of a block's four
// slices of K and the barriers between them; 17 us at 4,096 rows, where the
// two products took 45 us with the partial tiles added by atomics.
__global__ void __launch_bounds__(256)
    WeightGradKernel(int B, BatchSplit split, const uint16_t *h1, const uint16_t *dz1h,
                     const uint16_t *dz2h, const uint8_t *codes, const uint16_t *embh,
                     float *w1_parts, float *w2_parts, const float *sums, int nsums, float *grad,
                     float *loss) {
  __shared__ GemmLds T;
  __shared__ uint4 emb[kCostAlphabet + 1];
  int block = blockIdx.x;
  const int w1 = kW1Tiles * split.w1_slices;
  auto store = [&](float *c, int cols, int mb, int nb, const float16_t &acc) {
#pragma unroll
    for (int r = 0; r < 16; ++r)
      c[(size_t)(mb + TileRow(r)) * cols + nb + TileCol()] = acc[r];
  };
  if (block < w1) {
    if (threadIdx.x <= kCostAlphabet)
      emb[threadIdx.x] = threadIdx.x < kCostAlphabet
                             ? reinterpret_cast<const uint4 *>(embh)[threadIdx.x]
                             : make_uint4(0, 0, 0, 0);
    __syncthreads();
    const int tile = block % kW1Tiles, slice = block / kW1Tiles;
    const int mb = tile / (kCostIn / kGemmTile) * kGemmTile,
              nb = tile % (kCostIn / kGemmTile) * kGemmTile;
    const int kb = slice * split.w1_rows, ke = min(B, kb + split.w1_rows);
    store(w1_parts + (size_t)slice * kCostH1 * kCostIn, kCostIn, mb, nb,
          GemmTile(T, ColumnOperand{dz1h, kCostH1}, EmbedOperand{codes, emb}, mb, nb, kb, ke));
    return;
  }
  block -= w1;
  if (block >= kW2Tiles * split.w2_slices) {
    __shared__ float part[3][64];
    const int c = (block - kW2Tiles * split.w2_slices) * 64 + (int)(threadIdx.x & 63);
    const int wave = threadIdx.x >> 6;
    float sum = 0.f;
    if (c < kSums) {
#pragma unroll 16
      for (int b = wave; b < nsums; b += 4) sum += sums[(size_t)b * kSums + c];
    }
    if (wave > 0) part[wave - 1][threadIdx.x & 63] = sum;
    __syncthreads();
    if (wave > 0 || c >= kSums) return;
    sum += (part[0][threadIdx.x] + part[1][threadIdx.x]) + part[2][threadIdx.x];
    if (c < kSumB1) grad[kOffEmbed + c] = sum;
    else if (c < kSumB2) grad[kOffB1 + c - kSumB1] = sum;
    else if (c < kSumLoss) grad[kOffB2 + c - kSumB2] = sum;
    else *loss += sum;
    return;
  }
  const int nb = block % kW2Tiles * kGemmTile, slice = block / kW2Tiles;
  const int kb = slice * split.w2_rows, ke = min(B, kb + split.w2_rows);
  store(w2_parts + (size_t)slice * kCostH2 * kCostH1, kCostH1, 0, nb,
        GemmTile(T, ColumnOperand{dz2h, kCostH2}, ColumnOperand{h1, kCostH1}, 0, nb, kb, ke));
}

// ---------------------------------------------------------------------------
// Training, third kernel: the gradient's partial sums, Adam and the bf16
// copies of the weights.
// ---------------------------------------------------------------------------
struct Adam {
  float *w, *m, *v;
  uint16_t *w1h, *w2h, *embh;
  Operands o;
  float lr, b1, b2, eps;
  // weight i's bf16 copies
  __device__ __forceinline__ void Copy(size_t i, float x) const {
    const uint16_t h = F2Bf(x);
    if (i < kOffW1) {
      embh[i] = h;
    } else if (i < kOffB1) {
      const int k = (int)(i - kOffW1), unit = k / kCostIn, in = k % kCostIn;
      w1h[k] = h;
      o.w1[OperandAt(unit, in, kCostIn)] = h;
      o.w1t[OperandAt(in, unit, kCostH1)] = h;
    } else if (i >= kOffW2 && i < kOffB2) {
      const int k = (int)(i - kOffW2), unit = k / kCostH1, hidden = k % kCostH1;
      w2h[k] = h;
      o.w2[OperandAt(unit, hidden, kCostH1)] = h;
      o.w2t[OperandAt(hidden, unit, kCostH2)] = h;
    }
  }
};

// c1, c2: the step's bias corrections; lr = 0: no update.  keep: the whole
// gradient is left in g (W1's and W2's are only summed here).
__global__ void __launch_bounds__(256)
    AdamKernel(size_t n, Adam a, float *g, BatchSplit split, const float *w1_parts,
               const float *w2_parts, float c1, float c2, int keep) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float gi;
  if (i >= kOffW1 && i < kOffB1) {
    gi = 0.f;
    for (int k = 0; k < split.w1_slices; ++k)
      gi += w1_parts[(size_t)k * kCostH1 * kCostIn + (i - kOffW1)];
    if (keep) g[i] = gi;
  } else if (i >= kOffW2 && i < kOffB2) {
    gi = 0.f;
    for (int k = 0; k < split.w2_slices; ++k)
      gi += w2_parts[(size_t)k * kCostH2 * kCostH1 + (i - kOffW2)];
    if (keep) g[i] = gi;
  } else {
    gi = g[i];
  }
  if (a.lr == 0.f) return;
  const float mi = a.b1 * a.m[i] + (1.f - a.b1) * gi;
  const float vi = a.b2 * a.v[i] + (1.f - a.b2) * gi * gi;
  a.m[i] = mi;
  a.v[i] = vi;
  const float x = a.w[i] - a.lr * (mi / c1) / (sqrtf(vi / c2) + a.eps);
  a.w[i] = x;
  a.Copy(i, x);
}

__global__ void ZeroFloatKernel(size_t n, float *p) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.f;
}

__global__ void CopyBf16Kernel(size_t n, Adam a) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a.Copy(i, a.w[i]);
}

inline unsigned Blocks(size_t n, unsigned t = 256) { return (unsigned)((n + t - 1) / t); }

// ---------------------------------------------------------------------------
// Inference: one persistent kernel on v_mfma_f32_32x32x16_bf16 runs all three
// layers per tile of seeds, so no activation leaves the CU.
//
// Operand layout of the 32x32x16 MFMA: lane l supplies A[row l % 32][k] and
// B[k][column l % 32] for k = 8 * (l / 32) + j, j < 8; accumulator register r
// of lane l holds C[8 * (r / 4) + 4 * (l / 32) + (r % 4)][l % 32].
//
// Layers are computed transposed (hidden unit = row, seed = column); each
// wave owns 32 seeds:
//   layer 1: C1[h][seed] = W1[h][:] . x[seed][:] in kHB row blocks of 32
//            units; A = W1 from LDS ([k/8][unit][8]), a 32nd of the inputs
//            (16 KB) per stage in two alternating buffers, the next
//            stage read into registers during this one's MFMAs and stored
//            into the other buffer; B = the residue embeddings (one 16-byte
//            LDS read);
//   layer 2: C2[n][seed] = W2[n][:] . h1[:][seed], whose B operand is the
//            lane's own layer-1 accumulators (a lane holds one seed's column):
//            K step t takes registers 8 (t % 2) .. 8 (t % 2) + 7 of row block
//            t / 2, i.e. hidden units 16 t + 8 (j / 4) + 4 (l / 32) + j % 4,
//            and W2's columns are staged in LDS in that order;
//   layer 3: each lane sums its 32 rows of C2 and adds its partner lane's.
// Rounding points are those of the training forward (bf16 h1, h2, w3).
// ---------------------------------------------------------------------------
static_assert(kCostH1 % 32 == 0 && kCostH2 == 64, "inference tiles: H1 in 32s, H2 = 64");
constexpr int kHB = kCostH1 / 32;                  // layer-1 row blocks
// Blocks of four waves and 66 KB of LDS, two per CU: their stage barriers
// are independent, so one block's GELU epilogue overlaps the other's MFMAs.
constexpr int kInferWaves = 4;
constexpr int kInferTile = kInferWaves * 32;       // seeds per block pass
constexpr int kStageIn = 32;                       // W1 inputs per stage (4 residues)
constexpr int kStages = kCostIn / kStageIn;        // 32
static_assert(kStageIn == 32, "a stage's residues are one 32-bit word of codes");
constexpr int kStageVec = kCostH1 * kStageIn / 8;  // 16-byte pieces per stage
constexpr int kPrefetch = kStageVec / (kInferWaves * 64);
static_assert(kStageVec % (kInferWaves * 64) == 0, "a stage splits evenly over the block");
static_assert(kStages % 2 == 0, "stages alternate between two buffers across tiles");
static_assert((kStages & (kStages - 1)) == 0 && kStages * 4 == kCostResidues,
              "a row is kStages words; rotations wrap with a mask");
constexpr int kL2Steps = kCostH1 / 16;             // layer-2 K steps

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ bf16x8 Load8(const uint16_t *p) {
  return *reinterpret_cast<const bf16x8 *>(p);
}

__device__ __forceinline__ __bf16 AsBf16(uint16_t h) {
  return __builtin_bit_cast(__bf16, h);
}

// Piece i of stage s: unit h = i / 4, inputs s * 32 + (i % 4) * 8 .. + 8.
__device__ __forceinline__ uint4 StagePiece(const uint16_t *w1h, int s, int i) {
  const int h = i / (kStageIn / 8), k8 = i % (kStageIn / 8);
  return *reinterpret_cast<const uint4 *>(w1h + (size_t)h * kCostIn + s * kStageIn + k8 * 8);
}
__device__ __forceinline__ void PutPiece(uint16_t *w1s, int i, uint4 v) {
  const int h = i / (kStageIn / 8), k8 = i % (kStageIn / 8);
  *reinterpret_cast<uint4 *>(&w1s[(k8 * kCostH1 + h) * 8]) = v;
}

__global__ void __launch_bounds__(kInferWaves * 64) __attribute__((amdgpu_waves_per_eu(2)))
    InferKernel(const uint8_t *codes, uint32_t n, const uint32_t *count, uint32_t count_offset,
                const uint16_t *w1h, const uint16_t *embh, const float *b1, const uint16_t *w2h,
                const float *b2, const float *w3, const float *b3, uint32_t rotate, float *y) {
  // with `count`, the rows are the first *count - count_offset (at most n)
  if (count) {
    const uint32_t c = *count;
    n = c > count_offset ? min(n, c - count_offset) : 0u;
  }
  __shared__ __align__(16) uint16_t w1s[2][kStageIn * kCostH1];     // two stages, 32 KB
  __shared__ __align__(16) uint16_t w2[kL2Steps * 2 * 64 * 8];      // [t][row block][lane][8]
  __shared__ __align__(16) uint16_t emb[kCostAlphabet * kCostEmbed];
  __shared__ float b1s[kCostH1], b2s[kCostH2], w3s[kCostH2];
  for (int idx = threadIdx.x; idx < kL2Steps * 2 * 64 * 8; idx += blockDim.x) {
    const int j = idx & 7, l = (idx >> 3) & 63, nb = (idx >> 9) & 1, t = idx >> 10;
    const int row = 32 * nb + (l & 31);
    const int h = 16 * t + 8 * (j >> 2) + 4 * (l >> 5) + (j & 3);
    w2[idx] = w2h[row * kCostH1 + h];
  }
  for (int i = threadIdx.x; i < kCostAlphabet * kCostEmbed; i += blockDim.x) emb[i] = embh[i];
  for (int i = threadIdx.x; i < kCostH1; i += blockDim.x) b1s[i] = b1[i];
  if (threadIdx.x < kCostH2) {
    b2s[threadIdx.x] = b2[threadIdx.x];
    w3s[threadIdx.x] = Bf2F(F2Bf(w3[threadIdx.x]));
  }
  // stage 0 of W1; every later stage is read one stage ahead
#pragma unroll
  for (int p = 0; p < kPrefetch; ++p) {
    const int i = (int)threadIdx.x + p * kInferWaves * 64;
    PutPiece(w1s[0], i, StagePiece(w1h, 0, i));
  }
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int kq = lane >> 5, r32 = lane & 31;
  const uint32_t kshift = 8u * (uint32_t)kq;
  const float bias3 = b3[0];
  const uint32_t tiles = (n + kInferTile - 1) / kInferTile;
  for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    // the codes of this lane's seed stream through registers 4 at a time;
    // seeds past the end read seed 0's row as code 20 throughout
    const uint32_t seed = tile * kInferTile + wave * 32 + r32;
    const uint4 *src =
        reinterpret_cast<const uint4 *>(codes + (size_t)(seed < n ? seed : 0) * kCostResidues);
    const uint32_t fill = seed < n ? 0u : 0x14141414u;
    float16_t acc[kHB];
#pragma unroll
    for (int hb = 0; hb < kHB; ++hb)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[hb][r] = 0.f;
#pragma unroll 1
    for (int s = 0; s < kStages; ++s) {
      // stage s is in buffer s & 1; the next one (the first again after the
      // last; kStages is even) goes to the other buffer, which every wave
      // finished reading before the barrier that ended stage s - 1
      uint4 pf[kPrefetch];
      const int ns = (s + 1) % kStages;
#pragma unroll
      for (int p = 0; p < kPrefetch; ++p)
        pf[p] = StagePiece(w1h, ns, (int)threadIdx.x + p * kInferWaves * 64);
      const uint16_t *cur = w1s[s & 1];
      // residues 4 s .. 4 s + 3 of this lane's seed, the row read from word
      // `rotate` on (16 swaps its two halves of windows)
      const uint32_t cw =
          reinterpret_cast<const uint32_t *>(src)[(s + (int)rotate) & (kStages - 1)] | fill;
      // a K step's operands are read as one batch, a step ahead of its
      // MFMAs (the scheduling barriers keep that order), so the LDS latency
      // overlaps the previous step's MFMAs
      bf16x8 a[2][kHB], bx[2];
      auto load_step = [&](int q, bf16x8 (&av)[kHB], bf16x8 &b) {
        // residue 4 s + 2 q + kq: byte 2 q + kq of the word
        const int k8 = 2 * q + kq;
        uint32_t code = (cw >> (16 * q + kshift)) & 0xffu;
        code = code < 20 ? code : 20;
        b = Load8(&emb[code * kCostEmbed]);
#pragma unroll
        for (int hb = 0; hb < kHB; ++hb) av[hb] = Load8(&cur[(k8 * kCostH1 + 32 * hb + r32) * 8]);
      };
      load_step(0, a[0], bx[0]);
#pragma unroll
      for (int q = 0; q < kStageIn / 16; ++q) {
        if (q + 1 < kStageIn / 16) load_step(q + 1, a[(q + 1) & 1], bx[(q + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int hb = 0; hb < kHB; ++hb)
          acc[hb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[q & 1][hb], bx[q & 1], acc[hb],
                                                            0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int p = 0; p < kPrefetch; ++p)
        PutPiece(w1s[ns & 1], (int)threadIdx.x + p * kInferWaves * 64, pf[p]);
      __syncthreads();
    }
    float16_t acc2[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc2[0][r] = 0.f;
      acc2[1][r] = 0.f;
    }
#pragma unroll
    for (int t = 0; t < kL2Steps; ++t) {
      bf16x8 bh;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int h = 16 * t + 8 * (j >> 2) + 4 * kq + (j & 3);
        bh[j] = AsBf16(F2Bf(Gelu(acc[t >> 1][8 * (t & 1) + j] + b1s[h])));
      }
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        const bf16x8 a = Load8(&w2[((t * 2 + nb) * 64 + lane) * 8]);
        acc2[nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, bh, acc2[nb], 0, 0, 0);
      }
    }
    float part = 0.f;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 32 * nb + 8 * (r >> 2) + 4 * kq + (r & 3);
        part += Bf2F(F2Bf(Gelu(acc2[nb][r] + b2s[row]))) * w3s[row];
      }
    part += __shfl_xor(part, 32, 64);
    if (kq == 0 && seed < n) y[seed] = part + bias3;
  }
}

// Slices of the batch for a weight gradient, each of at least 256 rows; and a
// slice's rows, in whole K steps.
inline void SplitBatch(int B, int most, int *slices, int *rows) {
  most = std::max(1, std::min(most, B / 256));
  *rows = ((B + most - 1) / most + kGemmK - 1) / kGemmK * kGemmK;
  *slices = (B + *rows - 1) / *rows;
}

inline BatchSplit SplitOf(size_t B) {
  BatchSplit s;
  SplitBatch((int)B, kMostW1Slices, &s.w1_slices, &s.w1_rows);
  SplitBatch((int)B, kMostW2Slices, &s.w2_slices, &s.w2_rows);
  return s;
}

}  // namespace

// One allocation for several arrays, each on a 256-byte boundary.
class Slab {
 public:
  template <typename T>
  void Add(T **p, size_t count) {
    parts_[n_++] = {(void **)p, bytes_};
    bytes_ += (count * sizeof(T) + 255) / 256 * 256;
  }
  size_t bytes() const { return bytes_; }
  void Place(void *base) const {
    for (int i = 0; i < n_; ++i) *parts_[i].p = (char *)base + parts_[i].at;
  }

 private:
  struct Part {
    void **p;
    size_t at;
  };
  Part parts_[8];  // the most that a slab has
  int n_ = 0;
  size_t bytes_ = 0;
};

MlpDevice::MlpDevice() {
  count_ = kFlat;
  hipError_t e = hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking);
  Slab slab;
  slab.Add(&master_, kFlat);
  slab.Add(&grad_, kFlat + 1);  // and the loss
  slab.Add(&m_, kFlat);
  slab.Add(&v_, kFlat);
  slab.Add(&w1h_, (size_t)kCostH1 * kCostIn);
  slab.Add(&w2h_, (size_t)kCostH2 * kCostH1);
  slab.Add(&embh_, (size_t)kCostAlphabet * kCostEmbed);
  slab.Add(&operands_, (size_t)2 * kCostH1 * (kCostIn + kCostH2));
  if (e == hipSuccess) e = gz::Malloc(&weights_, slab.bytes());
  if (e == hipSuccess) slab.Place(weights_);
  init_status_ = e;
}

MlpDevice::~MlpDevice() {
  if (weights_) (void)gz::Free(weights_);
  if (batch_) (void)gz::Free(batch_);
  if (stream_) (void)hipStreamDestroy(stream_);
}

namespace {

Operands OperandsIn(uint16_t *p) {
  constexpr size_t kW1 = (size_t)kCostH1 * kCostIn, kW2 = (size_t)kCostH2 * kCostH1;
  return {p, p + kW1, p + 2 * kW1, p + 2 * kW1 + kW2};
}

Adam AdamOf(float *w, float *m, float *v, uint16_t *w1h, uint16_t *w2h, uint16_t *embh,
            uint16_t *operands, float lr) {
  return {w, m, v, w1h, w2h, embh, OperandsIn(operands), lr, 0.9f, 0.999f, 1e-8f};
}

}  // namespace

hipError_t MlpDevice::SetWeights(const CostModelWeights &w) {
  if (init_status_ != hipSuccess) return init_status_;
  std::vector<float> flat(kFlat);
  float *f = flat.data();
  auto put = [&](const std::vector<float> &v, size_t off) { memcpy(f + off, v.data(), v.size() * 4); };
  put(w.embed, kOffEmbed);
  put(w.w1, kOffW1);
  put(w.b1, kOffB1);
  put(w.w2, kOffW2);
  put(w.b2, kOffB2);
  put(w.w3, kOffW3);
  put(w.b3, kOffB3);
  hipError_t e = hipMemcpyAsync(master_, flat.data(), kFlat * 4, hipMemcpyHostToDevice, stream_);
  if (e == hipSuccess) e = hipMemsetAsync(m_, 0, kFlat * 4, stream_);
  if (e == hipSuccess) e = hipMemsetAsync(v_, 0, kFlat * 4, stream_);
  step_ = 0;
  if (e == hipSuccess) {
    hipLaunchKernelGGL(CopyBf16Kernel, dim3(Blocks(kFlat)), dim3(256), 0, stream_, kFlat,
                       AdamOf(master_, m_, v_, w1h_, w2h_, embh_, operands_, 0.f));
    e = hipGetLastError();
  }
  const hipError_t e2 = hipStreamSynchronize(stream_);
  return e != hipSuccess ? e : e2;
}

hipError_t MlpDevice::GetWeights(CostModelWeights *w) {
  if (init_status_ != hipSuccess) return init_status_;
  std::vector<float> flat(kFlat);
  const hipError_t e = hipMemcpy(flat.data(), master_, kFlat * 4, hipMemcpyDeviceToHost);
  if (e != hipSuccess) return e;
  auto get = [&](std::vector<float> &v, size_t off, size_t n) {
    v.assign(flat.begin() + off, flat.begin() + off + n);
  };
  get(w->embed, kOffEmbed, (size_t)kCostAlphabet * kCostEmbed);
  get(w->w1, kOffW1, (size_t)kCostH1 * kCostIn);
  get(w->b1, kOffB1, kCostH1);
  get(w->w2, kOffW2, (size_t)kCostH2 * kCostH1);
  get(w->b2, kOffB2, kCostH2);
  get(w->w3, kOffW3, kCostH2);
  get(w->b3, kOffB3, 1);
  return hipSuccess;
}

hipError_t MlpDevice::Reserve(size_t batch) {
  if (init_status_ != hipSuccess) return init_status_;
  if (batch <= cap_) return hipSuccess;
  cap_ = 0;
  if (batch_) (void)gz::Free(batch_);
  batch_ = nullptr;
  Slab slab;
  slab.Add(&codes_, batch * kCostResidues);
  slab.Add(&h1_, batch * kCostH1);
  slab.Add(&t_, batch);
  slab.Add(&dz2h_, batch * kCostH2);
  slab.Add(&dz1h_, batch * kCostH1);
  slab.Add(&w1_parts_, (size_t)kMostW1Slices * kCostH1 * kCostIn);
  slab.Add(&w2_parts_, (size_t)kMostW2Slices * kCostH2 * kCostH1);
  slab.Add(&sums_, (size_t)kMostBatchBlocks * kSums);
  const hipError_t e = gz::Malloc(&batch_, slab.bytes());
  if (e != hipSuccess) {
    batch_ = nullptr;
    return e;
  }
  slab.Place(batch_);
  cap_ = batch;
  return hipSuccess;
}

hipError_t MlpDevice::InferDevice(const uint8_t *d_codes, size_t n, float *d_out,
                                  hipStream_t s, uint32_t rotate_words, const uint32_t *d_count,
                                  uint32_t count_offset) {
  if (init_status_ != hipSuccess) return init_status_;
  if (n == 0) return hipSuccess;
  if (n > 0xFFFFFFFFull - kInferTile) return hipErrorInvalidValue;
  int dev = 0, cus = 256;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  const uint32_t tiles = (uint32_t)((n + kInferTile - 1) / kInferTile);
  hipLaunchKernelGGL(InferKernel, dim3(std::min<unsigned>(tiles, 2u * (unsigned)cus)),
                     dim3(kInferWaves * 64), 0, s, d_codes, (uint32_t)n, d_count, count_offset,
                     w1h_, embh_, master_ + kOffB1, w2h_, master_ + kOffB2, master_ + kOffW3,
                     master_ + kOffB3, rotate_words & (kStages - 1), d_out);
  return hipGetLastError();
}

hipError_t MlpDevice::Forward(const uint8_t *codes, size_t n, float *out, uint32_t rotate_words) {
  last_forward_ms = 0;
  if (n == 0) return hipSuccess;
  uint8_t *d_codes = nullptr;
  float *d_out = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  hipError_t e = gz::Malloc((void **)&d_codes, n * kCostResidues);
  if (e == hipSuccess) e = gz::Malloc((void **)&d_out, n * 4);
  if (e == hipSuccess) e = hipEventCreate(&e0);
  if (e == hipSuccess) e = hipEventCreate(&e1);
  if (e == hipSuccess)
    e = hipMemcpyAsync(d_codes, codes, n * kCostResidues, hipMemcpyHostToDevice, stream_);
  if (e == hipSuccess) e = hipEventRecord(e0, stream_);
  if (e == hipSuccess) e = InferDevice(d_codes, n, d_out, stream_, rotate_words);
  if (e == hipSuccess) e = hipEventRecord(e1, stream_);
  if (e == hipSuccess) e = hipMemcpyAsync(out, d_out, n * 4, hipMemcpyDeviceToHost, stream_);
  if (e == hipSuccess) e = hipStreamSynchronize(stream_);
  float ms = 0;
  if (e == hipSuccess && hipEventElapsedTime(&ms, e0, e1) == hipSuccess) last_forward_ms = ms;
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (d_codes) (void)gz::Free(d_codes);
  if (d_out) (void)gz::Free(d_out);
  return e;
}

hipError_t MlpDevice::TrainStep(const uint8_t *codes, const float *targets, size_t n,
                                float lr, float *loss, float *flat_grad) {
  const size_t B = (n + 63) / 64 * 64;
  hipError_t e = Reserve(B);
  if (e != hipSuccess) return e;
  hipStream_t s = stream_;
  (void)hipMemsetAsync(codes_, 20, B * kCostResidues, s);
  (void)hipMemcpyAsync(codes_, codes, n * kCostResidues, hipMemcpyHostToDevice, s);
  (void)hipMemsetAsync(t_, 0, B * 4, s);
  (void)hipMemcpyAsync(t_, targets, n * 4, hipMemcpyHostToDevice, s);
  hipLaunchKernelGGL(ZeroFloatKernel, dim3(1), dim3(64), 0, s, (size_t)1, grad_ + kFlat);
  if (lr != 0.f) ++step_;
  e = StepOnDevice(codes_, t_, nullptr, n, B, lr, step_, grad_ + kFlat, true);
  if (e != hipSuccess) return e;
  if (loss) (void)hipMemcpyAsync(loss, grad_ + kFlat, 4, hipMemcpyDeviceToHost, s);
  if (flat_grad) (void)hipMemcpyAsync(flat_grad, grad_, kFlat * 4, hipMemcpyDeviceToHost, s);
  return hipStreamSynchronize(s);
}

hipError_t MlpDevice::TrainEpochs(const uint8_t *codes, const float *targets, size_t n,
                                  const uint32_t *order, size_t m, size_t batch, float lr,
                                  float *mean_loss, float *kernel_ms) {
  if (mean_loss) *mean_loss = 0.f;
  if (kernel_ms) *kernel_ms = 0.f;
  if (n == 0 || m == 0 || batch == 0) return hipSuccess;
  const size_t B = (batch + 63) / 64 * 64;
  hipError_t e = Reserve(B);
  if (e != hipSuccess) return e;
  hipStream_t s = stream_;
  uint8_t *d_codes = nullptr;
  float *d_t = nullptr, *d_sum = nullptr;
  uint32_t *d_order = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  Slab slab;
  slab.Add(&d_codes, n * kCostResidues);
  slab.Add(&d_t, n);
  slab.Add(&d_order, m);
  slab.Add(&d_sum, 1);
  void *set = nullptr;
  size_t capacity = 0;
  e = WorkspacePool::Take(slab.bytes(), &set, &capacity);
  if (e != hipSuccess) return e;
  slab.Place(set);
  if (e == hipSuccess) e = hipEventCreate(&e0);
  if (e == hipSuccess) e = hipEventCreate(&e1);
  if (e == hipSuccess)
    e = hipMemcpyAsync(d_codes, codes, n * kCostResidues, hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipMemcpyAsync(d_t, targets, n * 4, hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipMemcpyAsync(d_order, order, m * 4, hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipMemsetAsync(d_sum, 0, 4, s);
  if (e == hipSuccess) e = hipEventRecord(e0, s);
  // whole batches only (the remainder of the order is left out, as the
  // per-step loop of the callers does); the steps' three launches each are
  // queued ahead of the device
  const size_t steps = m / batch;
  for (size_t done = 0; e == hipSuccess && done < steps; ++done)
    e = StepOnDevice(d_codes, d_t, d_order + done * batch, batch, B, lr, step_ + (long)done + 1,
                     d_sum, false);
  if (e == hipSuccess) e = hipEventRecord(e1, s);
  float sum = 0.f;
  if (e == hipSuccess) e = hipMemcpyAsync(&sum, d_sum, 4, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e == hipSuccess) step_ += (long)steps;
  if (e == hipSuccess && mean_loss && steps) *mean_loss = sum / (float)steps;
  float ms = 0.f;
  if (e == hipSuccess && kernel_ms && hipEventElapsedTime(&ms, e0, e1) == hipSuccess)
    *kernel_ms = ms;
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (e != hipSuccess) (void)hipStreamSynchronize(s);  // nothing may still read the set
  WorkspacePool::Give(set, capacity);
  return e;
}

// One optimisation step on a batch of n rows (padded to B) of codes and
// targets, taken through order (may be null); the batch's loss is added to
// *loss, and with keep the gradient left in grad_.  step: Adam's, from 1.
// Nothing is read back.
hipError_t MlpDevice::StepOnDevice(const uint8_t *codes, const float *targets,
                                   const uint32_t *order, size_t n, size_t B, float lr, long step,
                                   float *loss, bool keep) {
  hipStream_t s = stream_;
  const BatchSplit split = SplitOf(B);
  const BatchRows rows = {codes, targets, order, (int)n};
  const int tiles = (int)(B / kRows), batch_blocks = std::min(tiles, kMostBatchBlocks);
  hipLaunchKernelGGL(BatchKernel, dim3((unsigned)batch_blocks), dim3(256), 0, s, rows, tiles,
                     embh_, OperandsIn(operands_), master_ + kOffB1, master_ + kOffB2,
                     master_ + kOffW3, master_ + kOffB3, codes_, h1_, dz2h_, dz1h_, sums_);
  const unsigned blocks = (unsigned)(kW1Tiles * split.w1_slices + kW2Tiles * split.w2_slices) +
                          (kSums + 63) / 64;
  hipLaunchKernelGGL(WeightGradKernel, dim3(blocks), dim3(256), 0, s, (int)B, split, h1_, dz1h_,
                     dz2h_, codes_, embh_, w1_parts_, w2_parts_, sums_, batch_blocks, grad_, loss);
  const Adam a = AdamOf(master_, m_, v_, w1h_, w2h_, embh_, operands_, lr);
  const float c1 = 1.f - std::pow(a.b1, (float)step), c2 = 1.f - std::pow(a.b2, (float)step);
  hipLaunchKernelGGL(AdamKernel, dim3(Blocks(kFlat)), dim3(256), 0, s, kFlat, a, grad_, split,
                     w1_parts_, w2_parts_, c1, c2, keep ? 1 : 0);
  return hipGetLastError();
}

}  // namespace gz

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
using namespace gz;

struct gz_mlp_s {
  MlpDevice dev;
};

extern "C" {

size_t gz_mlp_weight_count(void) { return kFlat; }

gz_status gz_mlp_create(const float *flat, size_t count, gz_mlp_t *out) {
  GZ_REQUIRE(out && flat && count == kFlat, "gz_mlp_create: bad weights");
  CostModelWeights w;
  const float *f = flat;
  auto take = [&](std::vector<float> &v, size_t n) {
    v.assign(f, f + n);
    f += n;
  };
  take(w.embed, (size_t)kCostAlphabet * kCostEmbed);
  take(w.w1, (size_t)kCostH1 * kCostIn);
  take(w.b1, kCostH1);
  take(w.w2, (size_t)kCostH2 * kCostH1);
  take(w.b2, kCostH2);
  take(w.w3, kCostH2);
  take(w.b3, 1);
  std::unique_ptr<gz_mlp_s> h(new gz_mlp_s());
  GZ_HIP_CHECK(h->dev.SetWeights(w));
  *out = h.release();
  return GZ_OK;
}

gz_status gz_mlp_init_weights(uint64_t seed, float *flat) {
  CostModelWeights w;
  w.Init(seed);
  float *f = flat;
  for (auto *v : {&w.embed, &w.w1, &w.b1, &w.w2, &w.b2, &w.w3, &w.b3}) {
    memcpy(f, v->data(), v->size() * 4);
    f += v->size();
  }
  return GZ_OK;
}

gz_status gz_mlp_destroy(gz_mlp_t h) {
  delete h;
  return GZ_OK;
}

gz_status gz_mlp_predict(gz_mlp_t h, const uint8_t *codes, size_t n, float *out,
                         float *kernel_ms) {
  GZ_REQUIRE(h && (n == 0 || (codes && out)), "gz_mlp_predict: null argument");
  GZ_HIP_CHECK(h->dev.Forward(codes, n, out));
  if (kernel_ms) *kernel_ms = h->dev.last_forward_ms;
  return GZ_OK;
}

gz_status gz_mlp_predict_swapped(gz_mlp_t h, const uint8_t *codes, size_t n, float *out) {
  GZ_REQUIRE(h && (n == 0 || (codes && out)), "gz_mlp_predict_swapped: null argument");
  GZ_HIP_CHECK(h->dev.Forward(codes, n, out, kCostResidues / 8));
  return GZ_OK;
}

gz_status gz_mlp_train_step(gz_mlp_t h, const uint8_t *codes, const float *targets, size_t n,
                            float lr, float *loss, float *flat_grad) {
  GZ_REQUIRE(h && codes && targets && n > 0, "gz_mlp_train_step: bad argument");
  GZ_HIP_CHECK(h->dev.TrainStep(codes, targets, n, lr, loss, flat_grad));
  return GZ_OK;
}

gz_status gz_mlp_train_epochs(gz_mlp_t h, const uint8_t *codes, const float *targets, size_t n,
                              const uint32_t *order, size_t order_length, size_t batch, float lr,
                              float *mean_loss, float *kernel_ms) {
  GZ_REQUIRE(h && codes && targets && order && n > 0 && batch > 0,
             "gz_mlp_train_epochs: bad argument");
  for (size_t i = 0; i < order_length; ++i)
    GZ_REQUIRE(order[i] < n, "gz_mlp_train_epochs: order index out of range");
  GZ_HIP_CHECK(h->dev.TrainEpochs(codes, targets, n, order, order_length, batch, lr, mean_loss,
                                  kernel_ms));
  return GZ_OK;
}

gz_status gz_mlp_get_weights(gz_mlp_t h, float *flat) {
  GZ_REQUIRE(h && flat, "null argument");
  CostModelWeights w;
  GZ_HIP_CHECK(h->dev.GetWeights(&w));
  float *f = flat;
  for (auto *v : {&w.embed, &w.w1, &w.b1, &w.w2, &w.b2, &w.w3, &w.b3}) {
    memcpy(f, v->data(), v->size() * 4);
    f += v->size();
  }
  return GZ_OK;
}

gz_status gz_cost_features_packed_async(const uint64_t *pq, const uint64_t *pd,
                                        const uint32_t *qpos, const uint32_t *dpos, size_t n,
                                        int reverse, uint8_t *out, gz_stream_t stream) {
  GZ_REQUIRE(n < (1ull << 32), "gz_cost_features_packed_async: too many seeds");
  GZ_HIP_CHECK(CostFeaturesOnDevice(pq, pd, qpos, dpos, (uint32_t)n, reverse != 0, out,
                                    stream ? stream->s : nullptr));
  return GZ_OK;
}

void gz_cost_features(const uint8_t *queries, const uint8_t *database, const uint32_t *qpos,
                      const uint32_t *dpos, size_t n, int reverse, uint8_t *out) {
  for (size_t i = 0; i < n; ++i)
    CostFeatures(queries, database, qpos[i], dpos[i], reverse != 0, out + i * kCostResidues);
}

}  // extern "C"
