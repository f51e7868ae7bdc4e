// Learned SDF surrogate of the terrain field: training-data kernels (signed
// Euclidean distance transform of the field's zero set, point sampler), the
// fused MFMA forward/backward training kernel, the Adam + operand-packing
// kernel, and batched inference.  No reference counterpart; the CPU oracle's
// FP64 forward/backward checks these kernels.
//
// MFMA layout and the register chaining of layers: csrc/mlp_layout.hpp.
#include "../device_paths.hpp"
#include "../mlp_layout.hpp"

namespace re {
namespace {

using namespace mlp;

// Work-group size of the kernels that stage the network in LDS (42 KB per
// group): 8 waves share one copy, so LDS allows 3 groups = 24 waves per CU
// and the register budget, not LDS, sets the occupancy.
constexpr int kSurrBlock = 512;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// sin(2 pi x) and cos(2 pi x): v_sin_f32 / v_cos_f32 take the angle in
// revolutions; the argument is reduced to [0, 1) first.
__device__ __forceinline__ float sin_rev(float x) { return __builtin_amdgcn_sinf(__builtin_amdgcn_fractf(x)); }
__device__ __forceinline__ float cos_rev(float x) { return __builtin_amdgcn_cosf(__builtin_amdgcn_fractf(x)); }

// Hidden activation, SiLU: z * sigmoid(z), with sigmoid(z) =
// 1 / (1 + 2^(-z log2 e)) from the hardware exp2 and reciprocal (about 1 ulp
// each; the activations are rounded to BF16 anyway), not the IEEE division
// sequence.
__device__ __forceinline__ float sigmoid_fast(float z) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z * -1.44269504089f));
}
// The same unit on the scaled pre-activation u = -log2(e) z of the inference
// operands: u / (1 + 2^u) = -log2(e) SiLU(z).
__device__ __forceinline__ float silu_scaled(float u) { return u * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(u)); }

// Its derivative s (1 + z (1 - s)) from z and s = sigmoid(z).
__device__ __forceinline__ float dsilu(float z, float s) { return s * (1.0f + z * (1.0f - s)); }

// Device PCG32 (same generator as the host scene generators).
struct DevPcg {
  uint64_t state, inc;
  __device__ DevPcg(uint64_t initstate, uint64_t initseq) {
    state = 0u;
    inc = (initseq << 1u) | 1u;
    next();
    state += initstate;
    next();
  }
  __device__ uint32_t next() {
    uint64_t old = state;
    state = old * 6364136223846793005ULL + inc;
    uint32_t xs = (uint32_t)(((old >> 18u) ^ old) >> 27u);
    uint32_t rot = (uint32_t)(old >> 59u);
    return (xs >> rot) | (xs << ((32u - rot) & 31u));
  }
  __device__ float uniform() { return (float)(next() >> 8) * (1.0f / 16777216.0f); }
};

// ----------------------------------------------------------------- features

// The B operands of layer 0 for this lane's point: K-step c < 3 holds the
// sin/cos pairs of frequencies 4g..4g+3 of coordinate c (f_k = 2^(k/2), so
// f_{4g+2} = 2 f_{4g} and f_{4g+3} = 2 f_{4g+1}: those two pairs come from
// the double-angle identities, which keeps 4 of the 8 transcendentals);
// K-step 3 holds the raw coordinates (g = 0, s < 3) and zero padding.
__device__ __forceinline__ void features(f3 p, int g, bf16x8 xb[4]) {
  const float pc[3] = {p.x, p.y, p.z};
  const float f0 = (float)(1 << (2 * g));
  const float f1 = f0 * 1.41421356237f;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const float s0 = sin_rev(f0 * pc[c]), c0 = cos_rev(f0 * pc[c]);
    const float s1 = sin_rev(f1 * pc[c]), c1 = cos_rev(f1 * pc[c]);
    xb[c][0] = (__bf16)s0;
    xb[c][1] = (__bf16)c0;
    xb[c][2] = (__bf16)s1;
    xb[c][3] = (__bf16)c1;
    xb[c][4] = (__bf16)(2.0f * s0 * c0);
    xb[c][5] = (__bf16)((c0 - s0) * (c0 + s0));
    xb[c][6] = (__bf16)(2.0f * s1 * c1);
    xb[c][7] = (__bf16)((c1 - s1) * (c1 + s1));
  }
#pragma unroll
  for (int s = 0; s < 8; ++s) xb[3][s] = (__bf16)((g == 0 && s < 3) ? pc[s] : 0.0f);
}

// ----------------------------------------------------------------- forward

struct TileAct {
  f32x4 ds[4][4];   // dSiLU/dz [layer][M-tile], lane holds neurons 16m+4g+r (KEEP): kept instead of z, so that
                    // the backward pass takes no exponential and reciprocal of its own
  bf16x8 hb[4][2];  // bf16 B operands of h0..h3 (hb[3] feeds nothing but the staging)
  float h3[4][4];   // FP32 h3 for the output layer
};

template <bool KEEP, bool SCALED>
__device__ __forceinline__ float activate(float z, f32x4& ds, int r) {
  if (SCALED) return silu_scaled(z);
  const float s = sigmoid_fast(z);
  if (KEEP) ds[r] = dsilu(z, s);
  return z * s;
}

// SCALED: the inference operands (pre-activations carried as -log2(e) z).
template <bool KEEP, bool SCALED = false>
__device__ __forceinline__ float forward_tile(const bf16x8* __restrict__ packF, const float* __restrict__ small,
                                              const bf16x8 xb[4], int lane, TileAct& T) {
  const int g = lane >> 4;
  bf16x8 in[2];
  // layer 0: 4 K-steps of 32 features
  {
    f32x4 acc[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      acc[m] = *reinterpret_cast<const f32x4*>(&small[16 * m + 4 * g]);  // the bias starts the sum
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[m] = mfma16(packF[(oPackF0 >> 3) + (m * 4 + c) * 64 + lane], xb[c], acc[m]);
    }
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float z = acc[m][r];
        T.hb[0][m >> 1][(m & 1) * 4 + r] = (__bf16)activate<KEEP, SCALED>(z, T.ds[0][m], r);
      }
  }
  // layers 1..3: 2 K-steps of 32 neurons, chained in registers
#pragma unroll
  for (int L = 1; L < 4; ++L) {
    in[0] = T.hb[L - 1][0];
    in[1] = T.hb[L - 1][1];
    const int off = (oPackF1 + (L - 1) * kPackL) >> 3;
    f32x4 acc[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      acc[m] = *reinterpret_cast<const f32x4*>(&small[64 * L + 16 * m + 4 * g]);
#pragma unroll
      for (int c = 0; c < 2; ++c) acc[m] = mfma16(packF[off + (m * 2 + c) * 64 + lane], in[c], acc[m]);
    }
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float z = acc[m][r];
        const float h = activate<KEEP, SCALED>(z, T.ds[L][m], r);
        T.hb[L][m >> 1][(m & 1) * 4 + r] = (__bf16)h;
        if (L == 3) T.h3[m][r] = h;
      }
  }
  // output: partial dot over this lane's 16 neurons, summed over the 4 groups
  float o = 0.0f;
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) o += small[256 + 16 * m + 4 * g + r] * T.h3[m][r];
  o += __shfl_xor(o, 16);
  o += __shfl_xor(o, 32);
  return o + small[320];
}

// Copies the packed forward operands (and optionally the backward ones) and
// the small parameters into LDS.
__device__ __forceinline__ void load_weights(const bf16x8* __restrict__ gpack, const float* __restrict__ gsmall,
                                             bf16x8* spack, float* ssmall, int n_vec) {
  for (int i = threadIdx.x; i < n_vec; i += blockDim.x) spack[i] = gpack[i];
  for (int i = threadIdx.x; i < kSmall; i += blockDim.x) ssmall[i] = gsmall[i];
  __syncthreads();
}

// ----------------------------------------------------------------- inference

__global__ void __launch_bounds__(512) mlp_infer_kernel(const bf16x8* __restrict__ gpack,
                                                        const float* __restrict__ gsmall,
                                                        const float* __restrict__ pts, int64_t n,
                                                        float* __restrict__ out) {
  __shared__ bf16x8 spack[oPackB1 >> 3];
  __shared__ __align__(16) float ssmall[kSmall];
  load_weights(gpack, gsmall, spack, ssmall, oPackB1 >> 3);
  const int lane = threadIdx.x & 63;
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int64_t n_waves = ((int64_t)gridDim.x * blockDim.x) >> 6;
  const int64_t tiles = (n + 15) / 16;
  for (int64_t tile = wave; tile < tiles; tile += n_waves) {
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");  // weight reads stay in the loop
    int64_t i = tile * 16 + (lane & 15);
    const int64_t ic = i < n ? i : n - 1;
    const f3 p{pts[3 * ic], pts[3 * ic + 1], pts[3 * ic + 2]};
    bf16x8 xb[4];
    features(p, lane >> 4, xb);
    TileAct T;
    const float o = forward_tile<false, true>(spack, ssmall, xb, lane, T);
    if (lane < 16 && i < n) out[i] = o;
  }
}

// ----------------------------------------------------------------- training

// A block's eight waves take two 64-point chunks at a time, waves 0-3 the first
// and waves 4-7 the second, 16 points each.  Every wave runs forward and
// backward on its tile; the weight gradients are products over the points, so
// layer by layer the waves stage the bf16 dZ of the layer and its input
// activations, transposed as [neuron][point], in LDS, and after a barrier each
// wave accumulates its own two of the layer's 16 result tiles (three or four of
// layer 0's 28) with K = points, and the bias gradients of two of the layers as
// the product with a column of ones.  The output layer's gradient is summed in
// registers, per lane over its own points, and reduced over lanes and waves
// once at the end.  Staging one layer at a time (two buffers, one barrier per
// layer) is what leaves the LDS room for eight waves beside the 64 KB of
// operands; with four waves and every layer staged at once a SIMD ran one wave
// and stood still through its chains of LDS reads, MFMAs and exponentials:
// 38.5 us per launch of 65,536 points, now 30.8.
//
// Additions keep the order of one chunk after the other: K runs over the first
// chunk's points, then the second's, and the output layer's per-lane sums of
// both chunks are kept by one half (neurons m = 0, 1 by the first, 2, 3 by the
// second), which the other hands its products through LDS (exchange).
//
// A round of the loop has four barriers, B3 to B0, one per layer.  What lies
// between the last access of one use of an LDS area and the first of the next:
//   dz1, in1          staged for layer 3 before B3, read after it     B2
//                     staged for layer 1 before B1, read after it     B0
//   dz0, in0[0..63]   staged for layer 2 before B2, read after it     B1
//                     staged for layer 0 before B0, read after it     B3 of the next round
//   in0[64..], tail   exchange written after B3, read after B2        B1
//                     staged for layer 0 before B0, read after it     B3 of the next round
// (A wave in the next round passes B3 only when every wave has left layer 0 of
// this one, so the exchange must not be written before B3.)  After the loop the
// final sums are written to dz1, whose last readers are behind B0.
constexpr int kChunkPts = 64;
constexpr int kPairPts = 2 * kChunkPts;
// Staged rows are padded by 16 bytes (136 bf16): the 16 rows of one MFMA operand
// read then cover all 64 LDS banks once, and the four neuron groups of a
// staging write fall in different banks.
constexpr int kRow = kPairPts + 8;
// Layer-0 inputs staged: the 99 used, padded to 7 column tiles of 16.
constexpr int kInStage = 112;
constexpr int kTrainBlock = 512;
constexpr int kHalfThreads = kTrainBlock / 2;
constexpr int kExchange = 18;  // per lane of a half: 8 + 8 products of the output layer, dout, loss

struct TrainLds {
  bf16x8 pack[kPack >> 3];            // 64 KB: forward and backward operands
  float small[kSmall + 3];
  __bf16 dz1[kH][kRow], in1[kH][kRow];        // staging of layers 3 and 1
  __bf16 dz0[kH][kRow], in0[kInStage][kRow];  // staging of layers 2 and 0
  unsigned char tail[kExchange * kHalfThreads * 4 - (kInStage - kH) * kRow * 2];  // the exchange's end
};
static_assert(sizeof(TrainLds) <= 160 * 1024, "one training block must fit the LDS of a CU");
static_assert(sizeof(__bf16) * kH * kRow >= sizeof(float) * (4 * kH + 8),
              "the final reduction reuses a staging buffer");
static_assert((kPack >> 3) % kTrainBlock == 0, "the operand pack is copied in whole rounds");

__device__ __forceinline__ int64_t train_sample_index(int64_t batch_start, int ch, int p_local, int64_t n_samples) {
  return (batch_start + (int64_t)ch * kChunkPts + p_local) % n_samples;
}

__global__ void __launch_bounds__(kTrainBlock) mlp_train_kernel(const bf16x8* __restrict__ gpack,
                                                                const float* __restrict__ gsmall,
                                                                const float4* __restrict__ samples, int64_t n_samples,
                                                                int64_t batch_start, int32_t batch, float over_weight,
                                                                float* __restrict__ partial) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  TrainLds& S = *reinterpret_cast<TrainLds*>(lds_raw);
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int half = wv >> 2;           // which chunk of the pair
  const int g = lane >> 4, j = lane & 15;
  const int p_local = 16 * (wv & 3) + j;
  const int p_row = kChunkPts * half + p_local;
  const int mi = wv >> 1, odd = wv & 1;  // result tiles: rows 16 mi, and the even or odd wave's columns
  const float inv_b = 1.0f / (float)batch;
  const int n_chunks = batch / kChunkPts;
  // Rows of lane values, over rows of in0 that only layer 0 stages
  float* const exchange = reinterpret_cast<float*>(&S.in0[kH][0]);
  const int xl = threadIdx.x & (kHalfThreads - 1);

  // The first chunk's sample is requested before the operand copy, and the
  // copy issues all of a thread's loads before its first LDS store.
  float4 smp_next = make_float4(0.f, 0.f, 0.f, 0.f);
  {
    const int c0 = (int)blockIdx.x + half * (int)gridDim.x;
    if (c0 < n_chunks) smp_next = samples[train_sample_index(batch_start, c0, p_local, n_samples)];
    constexpr int kPer = (kPack >> 3) / kTrainBlock;
    bf16x8 r[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) r[k] = gpack[threadIdx.x + kTrainBlock * k];
    for (int i = threadIdx.x; i < kSmall; i += kTrainBlock) S.small[i] = gsmall[i];
#pragma unroll
    for (int k = 0; k < kPer; ++k) S.pack[threadIdx.x + kTrainBlock * k] = r[k];
  }
  __syncthreads();

  // [layer][tile], layers 1-3 use two tiles; biases of layers 0 and 1 (even
  // waves) or 2 and 3 (odd waves)
  f32x4 acc[4][4], accb[2];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    if (a < 2) accb[a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // B operand of the bias product: column 0 all ones, the other columns zero
  bf16x8 ones;
#pragma unroll
  for (int s = 0; s < 8; ++s) ones[s] = (__bf16)(j == 0 ? 1.0f : 0.0f);
  // per lane, over its points and those of the other half's same lane: dout * h3
  // for neurons 16 m + 4 g + r, m = 2 half, 2 half + 1; dout and the loss (first
  // half, g == 0 lanes)
  float dw4r[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) dw4r[q] = 0.0f;
  float db4r = 0.0f, loss = 0.0f;

  for (int ch = blockIdx.x; ch < n_chunks; ch += 2 * gridDim.x) {
    const bool have = ch + half * (int)gridDim.x < n_chunks;    // this half's chunk exists
    const bool two = ch + (int)gridDim.x < n_chunks;            // both do
    const int k_steps = two ? kPairPts / 32 : kChunkPts / 32;
    const float4 smp = smp_next;
    {
      const int next = ch + (2 + half) * (int)gridDim.x;
      if (next < n_chunks) smp_next = samples[train_sample_index(batch_start, next, p_local, n_samples)];
    }
    TileAct T;
    float dz[4][4], own[8], give[8], dout = 0.0f, l = 0.0f;
    if (have) {
      bf16x8 xb[4];
      features(f3{smp.x, smp.y, smp.z}, g, xb);
      const float o = forward_tile<true>(S.pack, S.small, xb, lane, T);
      const float r = o - smp.w;
      const float wgt = r > 0.0f ? over_weight : 1.0f;
      dout = 2.0f * wgt * r * inv_b;
      l = wgt * r * r * inv_b;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const float lo = dout * T.h3[q >> 2][q & 3], hi = dout * T.h3[2 + (q >> 2)][q & 3];
        own[q] = half ? hi : lo;
        give[q] = half ? lo : hi;
      }
      if (half == 0 && g == 0) {
        loss += l;
        db4r += dout;
      }
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int r2 = 0; r2 < 4; ++r2) dz[m][r2] = dout * S.small[256 + 16 * m + 4 * g + r2] * T.ds[3][m][r2];
    }

    // backward through the hidden layers, chaining dZ in registers
#pragma unroll
    for (int L = 3; L >= 0; --L) {
      __bf16(*const dzT)[kRow] = (L & 1) ? S.dz1 : S.dz0;
      __bf16(*const inT)[kRow] = (L & 1) ? S.in1 : S.in0;
      if (have) {
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
          for (int r2 = 0; r2 < 4; ++r2) dzT[16 * m + 4 * g + r2][p_row] = (__bf16)dz[m][r2];
        if (L > 0) {
#pragma unroll
          for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int r2 = 0; r2 < 4; ++r2)
              inT[16 * m + 4 * g + r2][p_row] = T.hb[L - 1][m >> 1][(m & 1) * 4 + r2];
        } else {
          // taken again (12 of the chunk's transcendentals): kept since the
          // forward pass they are 16 registers that the others then spill
          float px = smp.x, py = smp.y, pz = smp.z;
          asm volatile("" : "+v"(px), "+v"(py), "+v"(pz));
          bf16x8 xb[4];
          features(f3{px, py, pz}, g, xb);
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            if (c == 3 && g >= 2) break;  // rows 112..127 are zero padding, never read
#pragma unroll
            for (int s = 0; s < 8; ++s) inT[32 * c + 8 * g + s][p_row] = xb[c][s];
          }
        }
      }
      __syncthreads();  // barrier L of the table above
      if (L == 3 && have) {
#pragma unroll
        for (int q = 0; q < 8; ++q) exchange[(8 * half + q) * kHalfThreads + xl] = give[q];
        if (half == 1) {
          exchange[16 * kHalfThreads + xl] = dout;
          exchange[17 * kHalfThreads + xl] = l;
        }
      }
      if (L == 2) {
        // the first chunk's products, then the second's
        if (half == 0) {
#pragma unroll
          for (int q = 0; q < 8; ++q) dw4r[q] += own[q];
          if (two) {
#pragma unroll
            for (int q = 0; q < 8; ++q) dw4r[q] += exchange[(8 + q) * kHalfThreads + xl];
            if (g == 0) {
              db4r += exchange[16 * kHalfThreads + xl];
              loss += exchange[17 * kHalfThreads + xl];
            }
          }
        } else {
#pragma unroll
          for (int q = 0; q < 8; ++q) dw4r[q] += exchange[q * kHalfThreads + xl];
          if (two) {
#pragma unroll
            for (int q = 0; q < 8; ++q) dw4r[q] += own[q];
          }
        }
      }
      // this wave's tiles of dW = dZ^T (64 x points) . H (points x in)
      const int n0 = L > 0 ? 2 * odd : 4 * odd;  // first column tile
      const int n_tiles = L > 0 ? 2 : (odd ? 3 : 4);
#pragma unroll
      for (int kc = 0; kc < kPairPts / 32; ++kc) {
        if (kc >= k_steps) break;
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(&dzT[16 * mi + j][32 * kc + 8 * g]);
        if (odd == (L >> 1)) accb[L & 1] = mfma16(a, ones, accb[L & 1]);
#pragma unroll
        for (int t = 0; t < (L > 0 ? 2 : 4); ++t) {
          if (t >= n_tiles) break;
          acc[L][t] = mfma16(a, *reinterpret_cast<const bf16x8*>(&inT[16 * (n0 + t) + j][32 * kc + 8 * g]), acc[L][t]);
        }
      }
      if (have && L > 0) {
        bf16x8 dzb[2];
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
          for (int r2 = 0; r2 < 4; ++r2) dzb[m >> 1][(m & 1) * 4 + r2] = (__bf16)dz[m][r2];
        const int off = (oPackB1 + (L - 1) * kPackL) >> 3;
        f32x4 dh[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          dh[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int c = 0; c < 2; ++c) dh[m] = mfma16(S.pack[off + (m * 2 + c) * 64 + lane], dzb[c], dh[m]);
        }
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
          for (int r2 = 0; r2 < 4; ++r2) dz[m][r2] = dh[m][r2] * T.ds[L - 1][m][r2];
      }
    }
  }

  // write this block's partial gradient (flat parameter layout) and loss
  float* P = partial + (int64_t)blockIdx.x * (kParams + 1);
#pragma unroll
  for (int L = 0; L < 4; ++L) {
    const int nin = L == 0 ? kIn : kH;
    const int oW = L == 0 ? oW0 : (L == 1 ? oW1 : (L == 2 ? oW2 : oW3));
    const int ob = L == 0 ? ob0 : (L == 1 ? ob1 : (L == 2 ? ob2 : ob3));
    const int n0 = L > 0 ? 2 * odd : 4 * odd;
    const int n_tiles = L > 0 ? 2 : (odd ? 3 : 4);
    if (odd == (L >> 1) && j == 0)
#pragma unroll
      for (int r2 = 0; r2 < 4; ++r2) P[ob + 16 * mi + 4 * g + r2] = accb[L & 1][r2];
#pragma unroll
    for (int t = 0; t < (L > 0 ? 2 : 4); ++t) {
      if (t >= n_tiles) break;
#pragma unroll
      for (int r2 = 0; r2 < 4; ++r2) {
        const int i = 16 * mi + 4 * g + r2, k = 16 * (n0 + t) + j;
        if (k < nin) P[oW + i * nin + k] = acc[L][t][r2];
      }
    }
  }
  // the output layer: over the 16 points of a lane group, then over the four
  // waves of a half (the buffer of layers 3 and 1 has no readers left: every
  // wave has passed layer 0's barrier since)
  float* red = reinterpret_cast<float*>(&S.dz1[0][0]);  // [wave][64], then [wave][2]
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    float v = dw4r[q];
    v += __shfl_xor(v, 1);
    v += __shfl_xor(v, 2);
    v += __shfl_xor(v, 4);
    v += __shfl_xor(v, 8);
    if (j == 0) red[(wv & 3) * 64 + 16 * (2 * half + (q >> 2)) + 4 * g + (q & 3)] = v;
  }
  if (half == 0) {
    float d4 = db4r, l = loss;
    for (int off = 32; off > 0; off >>= 1) {
      d4 += __shfl_xor(d4, off);
      l += __shfl_xor(l, off);
    }
    if (lane == 0) {
      red[4 * 64 + 2 * wv] = d4;
      red[4 * 64 + 2 * wv + 1] = l;
    }
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const int n = threadIdx.x;
    P[oW4 + n] = red[n] + red[64 + n] + red[128 + n] + red[192 + n];
    if (n == 0) {
      P[ob4] = red[256] + red[258] + red[260] + red[262];
      P[kParams] = red[257] + red[259] + red[261] + red[263];
    }
  }
}

// Sum of the blocks' partial gradients; optionally an Adam step
// (Kingma & Ba 2015) on the FP32 master parameters; then the bf16 operand
// pack and FP32 small parameters are rewritten from the parameters.
__device__ __forceinline__ void pack_param(int p, float wv, __bf16* pack, float* small) {
  if (p < ob0) {  // W0
    const int i = p / kIn, k = p % kIn;
    const int m = i >> 4, c = k >> 5, gg = (k & 31) >> 3, s = k & 7;
    pack[oPackF0 + pack_index(m, c, 4, 16 * gg + (i & 15), s)] = (__bf16)wv;
    pack[oPackInfer + oPackF0 + pack_index(m, c, 4, 16 * gg + (i & 15), s)] = (__bf16)(wv * kNegLog2e);
    return;
  }
  const int oWs[3] = {oW1, oW2, oW3}, obs[4] = {ob0, ob1, ob2, ob3};
  for (int L = 0; L < 4; ++L)
    if (p >= obs[L] && p < obs[L] + kH) {
      small[64 * L + (p - obs[L])] = wv;
      small[oSmallInfer + 64 * L + (p - obs[L])] = wv * kNegLog2e;
      return;
    }
  for (int L = 1; L < 4; ++L)
    if (p >= oWs[L - 1] && p < oWs[L - 1] + kH * kH) {
      const int i = (p - oWs[L - 1]) / kH, k = (p - oWs[L - 1]) % kH;
      int gg, s;
      kperm_inv(k & 31, gg, s);
      pack[oPackF1 + (L - 1) * kPackL + pack_index(i >> 4, k >> 5, 2, 16 * gg + (i & 15), s)] = (__bf16)wv;
      pack[oPackInfer + oPackF1 + (L - 1) * kPackL + pack_index(i >> 4, k >> 5, 2, 16 * gg + (i & 15), s)] = (__bf16)wv;
      kperm_inv(i & 31, gg, s);
      pack[oPackB1 + (L - 1) * kPackL + pack_index(k >> 4, i >> 5, 2, 16 * gg + (k & 15), s)] = (__bf16)wv;
      return;
    }
  if (p >= oW4 && p < oW4 + kH) {
    small[256 + (p - oW4)] = wv;
    small[oSmallInfer + 256 + (p - oW4)] = wv * kNegLn2;
  } else if (p == ob4) {
    small[320] = wv;
    small[oSmallInfer + 320] = wv;
  }
}

// First stage of the sum over blocks: row kFold * s of the partial-gradient
// array receives the sum of rows kFold * s .. kFold * s + kFold - 1, each
// column by one thread (fixed order, so the result is deterministic).
constexpr int kFold = 16;

__global__ void partial_fold_kernel(float* __restrict__ partial, int32_t n_blocks) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p > kParams) return;
  const int b0 = blockIdx.y * kFold;
  const int b1 = b0 + kFold < n_blocks ? b0 + kFold : n_blocks;
  float acc = 0.0f;
  for (int b = b0; b < b1; ++b) acc += partial[(int64_t)b * (kParams + 1) + p];
  partial[(int64_t)b0 * (kParams + 1) + p] = acc;
}

__global__ void mlp_update_kernel(float* __restrict__ params, float* __restrict__ m1, float* __restrict__ m2,
                                  const float* __restrict__ partial, int32_t n_blocks, int32_t step, float lr,
                                  float b1, float b2, float eps, int32_t do_adam, float* __restrict__ grad_out,
                                  __bf16* __restrict__ pack, float* __restrict__ small, float* __restrict__ loss_out) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p > kParams) return;
  float gsum = 0.0f;
  if (partial)
    for (int b = 0; b < n_blocks; b += kFold) gsum += partial[(int64_t)b * (kParams + 1) + p];
  if (p == kParams) {
    if (loss_out) *loss_out = gsum;
    return;
  }
  if (grad_out) grad_out[p] = gsum;
  float wv = params[p];
  if (do_adam) {
    const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
    const float mm = b1 * m1[p] + (1.0f - b1) * gsum;
    const float vv = b2 * m2[p] + (1.0f - b2) * gsum * gsum;
    m1[p] = mm;
    m2[p] = vv;
    wv = wv - lr * (mm / c1) / (sqrtf(vv / c2) + eps);
    params[p] = wv;
  }
  pack_param(p, wv, pack, small);
}

// The two stages above in one launch: a block covers 64 parameters with
// kReduceRows rows of threads; row q sums the kFold-row groups q, q +
// kReduceRows, ... in row order, then one thread per parameter adds the group
// sums in group order and takes the Adam step.  Bound by the partials' 19.4 MB
// (256 blocks): with a row of threads per group every load is in flight at
// once, 7.6 us against 8.6 with four rows.  The additions are the ones the two stages make,
// in the same order, so the result is the same to the bit.
constexpr int kReduceParams = 64;
constexpr int kReduceRows = 16;
constexpr int kMaxFoldGroups = 64;

__global__ void __launch_bounds__(kReduceParams * kReduceRows) grad_reduce_update_kernel(
    float* __restrict__ params, float* __restrict__ m1, float* __restrict__ m2, const float* __restrict__ partial,
    int32_t n_blocks, int32_t step, float lr, float b1, float b2, float eps, int32_t do_adam,
    float* __restrict__ grad_out, __bf16* __restrict__ pack, float* __restrict__ small, float* __restrict__ loss_out) {
  __shared__ float gs[kMaxFoldGroups][kReduceParams];
  const int pl = threadIdx.x & (kReduceParams - 1), q = threadIdx.x / kReduceParams;
  const int p = blockIdx.x * kReduceParams + pl;
  const int n_groups = (n_blocks + kFold - 1) / kFold;
  if (p <= kParams) {
    for (int sg = q; sg < n_groups; sg += kReduceRows) {
      const int r0 = sg * kFold;
      const int r1 = r0 + kFold < n_blocks ? r0 + kFold : n_blocks;
      float v[kFold];
#pragma unroll
      for (int k = 0; k < kFold; ++k) v[k] = r0 + k < r1 ? partial[(int64_t)(r0 + k) * (kParams + 1) + p] : 0.0f;
      float acc = 0.0f;
#pragma unroll
      for (int k = 0; k < kFold; ++k)
        if (r0 + k < r1) acc += v[k];
      gs[sg][pl] = acc;
    }
  }
  __syncthreads();
  if (q != 0 || p > kParams) return;
  float gsum = 0.0f;
  for (int sg = 0; sg < n_groups; ++sg) gsum += gs[sg][pl];
  if (p == kParams) {
    if (loss_out) *loss_out = gsum;
    return;
  }
  if (grad_out) grad_out[p] = gsum;
  float wv = params[p];
  if (do_adam) {
    const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
    const float mm = b1 * m1[p] + (1.0f - b1) * gsum;
    const float vv = b2 * m2[p] + (1.0f - b2) * gsum * gsum;
    m1[p] = mm;
    m2[p] = vv;
    wv = wv - lr * (mm / c1) / (sqrtf(vv / c2) + eps);
    params[p] = wv;
  }
  pack_param(p, wv, pack, small);
}

// ----------------------------------------------------------------- training data

// Squared distance (voxel units) from each voxel to the zero set, seeded at
// voxels whose sign differs from a 6-neighbour with the linear-interpolation
// estimate of the sub-voxel distance; INF elsewhere.
__global__ void edt_seed_kernel(VolView V, float* __restrict__ g) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t n = (int64_t)V.dim[0] * V.dim[1] * V.dim[2];
  if (i >= n) return;
  const int x = (int)(i % V.dim[0]), y = (int)((i / V.dim[0]) % V.dim[1]), z = (int)(i / ((int64_t)V.dim[0] * V.dim[1]));
  const float f = V.data[vox_index(V.bdim, x, y, z)];
  float best = 1e20f;
  const int dx[6] = {1, -1, 0, 0, 0, 0}, dy[6] = {0, 0, 1, -1, 0, 0}, dz[6] = {0, 0, 0, 0, 1, -1};
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const int xn = x + dx[k], yn = y + dy[k], zn = z + dz[k];
    if (xn < 0 || yn < 0 || zn < 0 || xn >= V.dim[0] || yn >= V.dim[1] || zn >= V.dim[2]) continue;
    const float fn = V.data[vox_index(V.bdim, xn, yn, zn)];
    if ((f > 0.0f) != (fn > 0.0f)) {
      const float fr = fabsf(f) / fabsf(f - fn);
      best = fminf(best, fr * fr);
    }
  }
  g[i] = best;
}

// One separable pass of the exact Euclidean distance transform: for every
// line along `axis`, D(x) = min_x' (x - x')^2 + g(x').  One work-group per
// line; the line is staged in LDS (at most 4096 voxels).
__global__ void __launch_bounds__(256) edt_pass_kernel(const float* __restrict__ gin, float* __restrict__ gout,
                                                       int32_t dx, int32_t dy, int32_t dz, int32_t axis) {
  __shared__ float line[4096];
  const int64_t lid = blockIdx.x;
  int len, a, b;
  int64_t base, stride;
  if (axis == 0) { len = dx; a = (int)(lid % dy); b = (int)(lid / dy); base = ((int64_t)b * dy + a) * dx; stride = 1; }
  else if (axis == 1) { len = dy; a = (int)(lid % dx); b = (int)(lid / dx); base = (int64_t)b * dy * dx + a; stride = dx; }
  else { len = dz; a = (int)(lid % dx); b = (int)(lid / dx); base = (int64_t)b * dx + a; stride = (int64_t)dx * dy; }
  for (int x = threadIdx.x; x < len; x += blockDim.x) line[x] = gin[base + x * stride];
  __syncthreads();
  for (int x = threadIdx.x; x < len; x += blockDim.x) {
    float best = 1e20f;
    for (int q = 0; q < len; ++q) {
      const float d = (float)(x - q);
      best = fminf(best, d * d + line[q]);
    }
    gout[base + x * stride] = best;
  }
}

// Signed distance in world units, written into a bricked volume.
__global__ void edt_finish_kernel(VolView V, const float* __restrict__ g, float* __restrict__ out, float spacing) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t n = (int64_t)V.dim[0] * V.dim[1] * V.dim[2];
  if (i >= n) return;
  const int x = (int)(i % V.dim[0]), y = (int)((i / V.dim[0]) % V.dim[1]), z = (int)(i / ((int64_t)V.dim[0] * V.dim[1]));
  const int64_t vi = vox_index(V.bdim, x, y, z);
  const float f = V.data[vi];
  const float d = sqrtf(fminf(g[i], 1e12f)) * spacing;
  out[vi] = f > 0.0f ? d : -d;
}

// 2^k training points: even indices uniform in the volume, odd indices near
// the surface (|signed distance| < near_band, by bounded rejection).  Each
// sample is (x, y, z, signed distance).
template <bool NARROW>
__global__ void sample_kernel(VolView edt, float lo, float hi, int64_t n, uint64_t seed, float near_band,
                              int32_t max_tries, float4* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  DevPcg rng(seed, (uint64_t)i);
  f3 p{0, 0, 0};
  float d = 0.0f;
  const bool near = (i & 1) != 0;
  for (int t = 0; t < (near ? max_tries : 1); ++t) {
    p = f3{lo + (hi - lo) * rng.uniform(), lo + (hi - lo) * rng.uniform(), lo + (hi - lo) * rng.uniform()};
    d = trilinear<NARROW>(edt, p);
    if (!near || fabsf(d) < near_band) break;
  }
  out[i] = float4{p.x, p.y, p.z, d};
}

// ----------------------------------------------------------------- hybrid tracer

// Surrogate distance at the points of the lanes that need it.  The wave packs
// those points densely into its LDS slots (lane order), evaluates
// ceil(count / 16) tiles of 16 points, and each lane reads its result back,
// so a partly idle wave evaluates no empty tile rows.  LDS is in order within
// a wave; the fences keep the compiler from moving the slot reads and writes
// across each other.
__device__ __forceinline__ float wave_surrogate(const bf16x8* spack, const float* ssmall, f3 p, bool need,
                                                float* __restrict__ wpts, float* __restrict__ wout) {
  const int lane = threadIdx.x & 63;
  const unsigned long long mask = __ballot(need);
  const int count = __popcll(mask);
  const int slot = __popcll(mask & ((1ull << lane) - 1ull));
  if (need) {
    wpts[slot] = p.x;
    wpts[64 + slot] = p.y;
    wpts[128 + slot] = p.z;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll 1
  for (int q = 0; q < count; q += 16) {
    // keeps the weight reads inside the loop (hoisted, they would hold ~160
    // VGPRs for the whole kernel and cut occupancy to one wave per SIMD)
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int idx = q + (lane & 15);
    const int src = idx < count ? idx : count - 1;
    const f3 pq{wpts[src], wpts[64 + src], wpts[128 + src]};
    bf16x8 xb[4];
    features(pq, lane >> 4, xb);
    TileAct T;
    const float o = forward_tile<false, true>(spack, ssmall, xb, lane, T);
    if (lane < 16 && idx < count) wout[idx] = o;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  return need ? wout[slot] : 0.0f;
}

// The march through the learned distance, one ray per lane; a wave takes new
// rays for its idle lanes once half of its lanes are idle.
// Exact-phase march: h = max(f * k_exact, h_min) from a point with f > 0;
// on the first sample with f <= 0 the crossing is bisected (n_bisect steps)
// between the last positive and the first non-positive sample.
// Surrogate phase: step by (s - margin) while the surrogate distance s
// exceeds tau, then hand over to the exact phase; after rejoin of exact
// travel without a crossing, return to the surrogate.
constexpr int kDeferTile = 16;
// Blocks of the network's march: two per CU (84 VGPRs, 50 KB of LDS), each
// wave taking rays until the block's are gone.  With a block per 512 rays a
// block stayed until its longest march was done and whole blocks of the image
// cost many times others: 921,600 rays on 192^3 1,042 us, now 964 (their 7.7 M
// network points alone take 610 at the inference kernel's rate).  Times here
// and below are the kernel's alone, with one network trained for the sweep;
// another network evaluates another number of points.
constexpr int64_t kHybridBlocks = 512;
// Rays a wave holds: 64, or fewer while 12,288 runs (three per wave) are not
// reached, as a wave lasts as long as its longest march and the network's
// tile is 16 points.  us for 16 / 32 / 64 (and a block per 512 rays): 14,400
// rays 93 / 127 / 160 (198); 90,000 203 / 291 / 331 (323); 140,500 252 / 278 /
// 303 (334); 230,400 422 / 418 / 528 (487); 360,000 595 / 515 / 663 (596);
// 518,400 783 / 719 / 729 (763); 921,600 1,355 / 1,122 / 964 (1,042).
constexpr int64_t kHybridRuns = 12288;

template <bool USE_MLP, bool NARROW>
__global__ void __launch_bounds__(512) hybrid_trace_kernel(
    VolView V, float bx1, float by1, float bz1, const bf16x8* __restrict__ gpack, const float* __restrict__ gsmall,
    const float* __restrict__ ray_o, const float* __restrict__ ray_d, int64_t n, HybridParams hp,
    float* __restrict__ t_out, uint8_t* __restrict__ hit_out, int32_t* __restrict__ evals_out,
    int32_t* __restrict__ samples_out, int32_t log_lanes) {
  __shared__ bf16x8 spack[USE_MLP ? (oPackB1 >> 3) : 1];
  __shared__ __align__(16) float ssmall[kSmall];
  __shared__ float slots[USE_MLP ? kSurrBlock / 64 : 1][4 * 64];  // per wave: x, y, z, result
  __shared__ uint32_t queue;  // the block's rays taken so far
  if (USE_MLP) {
    if (threadIdx.x == 0) queue = 0u;
    load_weights(gpack, gsmall, spack, ssmall, oPackB1 >> 3);
  }
  const float bmin[3] = {0.0f, 0.0f, 0.0f}, bmax[3] = {bx1, by1, bz1};
  if (!USE_MLP) {
    // Without the network: the exact-field march from the volume entry.
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
      const f3 o{ray_o[3 * i], ray_o[3 * i + 1], ray_o[3 * i + 2]};
      const f3 d{ray_d[3 * i], ray_d[3 * i + 1], ray_d[3 * i + 2]};
      float t;
      int32_t samples;
      const bool h = exact_march<NARROW>(V, bmin, bmax, o, d, hp.k_exact, hp.h_min, hp.n_bisect, hp.max_iters, t, samples);
      t_out[i] = t;
      hit_out[i] = h ? 1 : 0;
      if (evals_out) evals_out[i] = 0;
      if (samples_out) samples_out[i] = samples;
    }
    return;
  }
  // The block's rays: every gridDim.x-th run of `lanes` from its own on.
  const int lanes = 1 << log_lanes;
  const int64_t runs = (n + lanes - 1) >> log_lanes;
  const uint32_t total = (uint32_t)((runs - blockIdx.x + gridDim.x - 1) / gridDim.x) << log_lanes;
  enum { SURR = 0, EXACT = 1, DONE = 2 };
  const int lane = threadIdx.x & 63;
  int phase = DONE;
  bool hit = false, drained = false;  // drained: wave-uniform
  int64_t ray = -1;
  f3 o{0, 0, 0}, d{0, 0, 0};
  float t = 0.0f, t_far = 0.0f, f_prev = 0.0f, travel = 0.0f;
  int32_t evals = 0, samples = 0, advances = 0;
  // A ray is advanced at most max_iters times (one network evaluation and/or
  // one exact step per advance).  While some lane can take an exact step, the
  // network only runs full 16-point tiles of the waiting lanes (which ones is
  // rotated from iteration to iteration); when none can, it runs for all of
  // them.  A waiting lane keeps its state, so every ray takes the same steps
  // as when the network runs for every waiting lane at once, in fewer
  // part-filled tiles.  Each wave iteration takes a ray, finds the queue empty
  // or advances at least one lane, which bounds the loop.
#pragma unroll 1
  for (uint32_t it = 0;; ++it) {
    if (phase != DONE && advances >= hp.max_iters) phase = DONE;
    const bool idle = phase == DONE;
    const unsigned long long imask = __ballot(idle && lane < lanes);
    const uint32_t want = (uint32_t)__popcll(imask);
    if (!drained && 2 * want >= (uint32_t)lanes) {
      if (idle && ray >= 0) {
        t_out[ray] = hit ? t : kInf;
        hit_out[ray] = hit ? 1 : 0;
        if (evals_out) evals_out[ray] = evals;
        if (samples_out) samples_out[ray] = samples;
        ray = -1;
      }
      const uint32_t at = (uint32_t)__builtin_amdgcn_readfirstlane((int)atomicAdd(&queue, lane == 0 ? want : 0u));
      drained = at + want >= total;
      const uint32_t s = at + (uint32_t)__popcll(imask & ((1ull << lane) - 1ull));
      const int64_t i = (((int64_t)blockIdx.x + (int64_t)(s >> log_lanes) * gridDim.x) << log_lanes) + (s & (uint32_t)(lanes - 1));
      if (idle && lane < lanes && s < total && i < n) {
        ray = i;
        o = f3{ray_o[3 * i], ray_o[3 * i + 1], ray_o[3 * i + 2]};
        d = f3{ray_d[3 * i], ray_d[3 * i + 1], ray_d[3 * i + 2]};
        hit = false;
        t = 0.0f;
        evals = samples = advances = 0;
        float tn, tf;
        if (ray_box(bmin, bmax, o, d, tn, tf)) {
          t = tn;
          t_far = tf;
          phase = SURR;
        }
      }
      continue;
    }
    if (want == (uint32_t)lanes) break;  // and drained: an idle wave takes rays as long as there are some
    bool advanced = phase == EXACT;
    const bool wait = phase == SURR;
    const unsigned long long wmask = __ballot(wait);
    const int n_wait = __popcll(wmask);
    const int n_run = __any(phase == EXACT) ? (n_wait & ~(kDeferTile - 1)) : n_wait;
    if (n_run > 0) {
      const int rank = __popcll(wmask & ((1ull << lane) - 1ull));
      const bool need = wait && (rank + (int)(it % (uint32_t)n_wait)) % n_wait < n_run;
      float* ws = slots[threadIdx.x >> 6];
      const float s = wave_surrogate(spack, ssmall, add(o, smul(t, d)), need, ws, ws + 192);
      if (need) {
        advanced = true;
        ++evals;
        if (s > hp.tau) {
          t += s - hp.margin;
          if (t >= t_far) phase = DONE;
        } else {
          phase = EXACT;
          travel = 0.0f;
          f_prev = trilinear<NARROW>(V, add(o, smul(t, d)));
          ++samples;
          if (f_prev <= 0.0f) {
            hit = true;  // entered the surface region already inside: accept the current point
            phase = DONE;
          }
        }
      }
    }
    if (phase == EXACT) {
      const float h = fmaxf(f_prev * hp.k_exact, hp.h_min);
      const float t_next = t + h;
      const float f_next = trilinear<NARROW>(V, add(o, smul(t_next, d)));
      ++samples;
      if (f_next <= 0.0f) {
        float a = t, b = t_next;
        for (int k = 0; k < hp.n_bisect; ++k) {
          const float mid = 0.5f * (a + b);
          const float fm = trilinear<NARROW>(V, add(o, smul(mid, d)));
          ++samples;
          if (fm > 0.0f) a = mid; else b = mid;
        }
        t = 0.5f * (a + b);
        hit = true;
        phase = DONE;
      } else {
        t = t_next;
        f_prev = f_next;
        travel += h;
        if (t >= t_far) phase = DONE;
        else if (travel > hp.rejoin) phase = SURR;
      }
    }
    if (advanced) ++advances;
  }
  if (ray >= 0) {
    t_out[ray] = hit ? t : kInf;
    hit_out[ray] = hit ? 1 : 0;
    if (evals_out) evals_out[ray] = evals;
    if (samples_out) samples_out[ray] = samples;
  }
}

}  // namespace

// ---------------------------------------------------------------- launchers

hipError_t launch_hybrid_trace(const DevVolume& field, const void* pack, const float* small, const float* ray_o,
                               const float* ray_d, int64_t n, const HybridParams& hp, bool use_mlp, float* t,
                               uint8_t* hit, int32_t* evals, int32_t* samples, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const VolView V = field.view();
  // Without the network one wave per block: a block's waves end together in
  // the scheduler's accounts, and marches differ many times in length (137 us
  // against 147 with blocks of 256 on 921,600 rays).
  const int block = use_mlp ? kSurrBlock : 64;
  int64_t blocks = (n + block - 1) / block;
  int32_t log_lanes = 6;
  if (use_mlp) {
    log_lanes = n <= 16 * kHybridRuns ? 4 : n <= 32 * kHybridRuns ? 5 : 6;
    const int64_t runs = (n + (1 << log_lanes) - 1) >> log_lanes;
    blocks = runs < kHybridBlocks ? runs : kHybridBlocks;
  }
#define RE_LAUNCH(MLP, NARROW)                                                                                     \
  hipLaunchKernelGGL((hybrid_trace_kernel<MLP, NARROW>), dim3((unsigned)blocks), dim3(block), 0, s,                \
                     V, field.box_max[0], field.box_max[1], field.box_max[2], (const bf16x8*)pack, small, ray_o,      \
                     ray_d, n, hp, t, hit, evals, samples, log_lanes)
  if (V.narrow) {
    if (use_mlp) RE_LAUNCH(true, true); else RE_LAUNCH(false, true);
  } else {
    if (use_mlp) RE_LAUNCH(true, false); else RE_LAUNCH(false, false);
  }
#undef RE_LAUNCH
  return hipGetLastError();
}

size_t mlp_train_lds_bytes() { return sizeof(TrainLds); }

hipError_t launch_mlp_infer(const void* pack, const float* small, const float* pts, int64_t n, float* out,
                            hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int64_t tiles = (n + 15) / 16;
  int64_t blocks = (tiles + kSurrBlock / 64 - 1) / (kSurrBlock / 64);
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(mlp_infer_kernel, dim3((unsigned)blocks), dim3(kSurrBlock), 0, s, (const bf16x8*)pack, small,
                     pts, n, out);
  return hipGetLastError();
}

hipError_t launch_mlp_train(const void* pack, const float* small, const float4* samples, int64_t n_samples,
                            int64_t batch_start, int32_t batch, float over_weight, float* partial, int32_t blocks,
                            hipStream_t s) {
  hipLaunchKernelGGL(mlp_train_kernel, dim3(blocks), dim3(kTrainBlock), sizeof(TrainLds), s, (const bf16x8*)pack, small,
                     samples, n_samples, batch_start, batch, over_weight, partial);
  return hipGetLastError();
}

hipError_t launch_mlp_update(float* params, float* m1, float* m2, float* partial, int32_t n_blocks,
                             int32_t step, float lr, float b1, float b2, float eps, int32_t do_adam, float* grad_out,
                             void* pack, float* small, float* loss_out, hipStream_t s) {
  const int threads = 256;
  const int blocks = (kParams + 1 + threads - 1) / threads;
  if (partial && n_blocks > 0 && (n_blocks + kFold - 1) / kFold <= kMaxFoldGroups) {
    hipLaunchKernelGGL(grad_reduce_update_kernel, dim3((kParams + kReduceParams) / kReduceParams),
                       dim3(kReduceParams * kReduceRows), 0, s,
                       params, m1, m2, partial, n_blocks, step, lr, b1, b2, eps, do_adam, grad_out, (__bf16*)pack,
                       small, loss_out);
    return hipGetLastError();
  }
  if (partial && n_blocks > 0)
    hipLaunchKernelGGL(partial_fold_kernel, dim3(blocks, (n_blocks + kFold - 1) / kFold), dim3(threads), 0, s,
                       partial, n_blocks);
  hipLaunchKernelGGL(mlp_update_kernel, dim3(blocks), dim3(threads), 0, s, params, m1, m2, partial, n_blocks, step,
                     lr, b1, b2, eps, do_adam, grad_out, (__bf16*)pack, small, loss_out);
  return hipGetLastError();
}

hipError_t launch_edt(const DevVolume& field, float* scratch_a, float* scratch_b, float* out_bricked,
                      hipStream_t s) {
  const VolView V = field.view();
  const int64_t n = (int64_t)V.dim[0] * V.dim[1] * V.dim[2];
  const int64_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(edt_seed_kernel, dim3((unsigned)blocks), dim3(256), 0, s, V, scratch_a);
  hipLaunchKernelGGL(edt_pass_kernel, dim3((unsigned)((int64_t)V.dim[1] * V.dim[2])), dim3(256), 0, s, scratch_a,
                     scratch_b, V.dim[0], V.dim[1], V.dim[2], 0);
  hipLaunchKernelGGL(edt_pass_kernel, dim3((unsigned)((int64_t)V.dim[0] * V.dim[2])), dim3(256), 0, s, scratch_b,
                     scratch_a, V.dim[0], V.dim[1], V.dim[2], 1);
  hipLaunchKernelGGL(edt_pass_kernel, dim3((unsigned)((int64_t)V.dim[0] * V.dim[1])), dim3(256), 0, s, scratch_a,
                     scratch_b, V.dim[0], V.dim[1], V.dim[2], 2);
  hipLaunchKernelGGL(edt_finish_kernel, dim3((unsigned)blocks), dim3(256), 0, s, V, scratch_b, out_bricked,
                     V.spacing[0]);
  return hipGetLastError();
}

hipError_t launch_sample(const DevVolume& edt, int64_t n, uint64_t seed, float near_band, int32_t max_tries,
                         float4* out, hipStream_t s) {
  const VolView V = edt.view();
  const float hi = (float)(V.dim[0] - 1) * V.spacing[0];
  const dim3 grid((unsigned)((n + 255) / 256));
  if (V.narrow)
    hipLaunchKernelGGL(sample_kernel<true>, grid, dim3(256), 0, s, V, 0.0f, hi, n, seed, near_band, max_tries, out);
  else
    hipLaunchKernelGGL(sample_kernel<false>, grid, dim3(256), 0, s, V, 0.0f, hi, n, seed, near_band, max_tries, out);
  return hipGetLastError();
}

}  // namespace re
