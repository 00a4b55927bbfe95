// Learned pilot-to-grid channel estimator: a 1-D convolutional network over the
// pilot positions of one (receive, transmit) stream pair, bfloat16 weights and
// activations on the MFMA units with float32 accumulation, and the kernels that
// train it on drops the simulator generates (backward-data on the same MFMA
// convolution, weight gradients, NMSE loss, Adam).
//
// Layout: sample s = (t * num_drops + d) * num_rx + r, positions p = 0..63,
// channels innermost: activations [S][64][C].  Weights [Cout][taps][Cin].  The
// positions are cyclic (a stream's pilots on a grid without DC roll sample the
// periodic frequency response uniformly), so every convolution is circular:
// out[p] = sum_k w[k] in[(p + (k - taps/2) dil) mod 64], with dilations 1, 4, 16, 1
// in the four layers (a receptive field covering the whole axis) and 1 in the skip.  The network is the learned counterpart of
// OrthogonalLeastSquaresChannelEstimation's interpolation
// (hermespy/modem/waveforms/orthogonal/channel.py:29-66): it maps the LS values at
// a stream's pilots to the channel of every resource element.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "hpx_common.hpp"

using namespace hpx;

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kPos = 64;   // pilot positions per sample
constexpr int kTaps = 5;       // the four layers
constexpr int kSkipTaps = 17;  // the linear skip convolution
constexpr int kDil1 = 1, kDil2 = 4, kDil3 = 16, kDil4 = 1;

inline hipStream_t as_stream(void* s) { return static_cast<hipStream_t>(s); }

__device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
  return static_cast<uint16_t>(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float(static_cast<uint32_t>(h) << 16); }

// GELU, tanh form
__device__ __forceinline__ float gelu(float x) {
  const float k0 = 0.7978845608028654f, k1 = 0.044715f;
  return 0.5f * x * (1.0f + tanhf(k0 * (x + k1 * x * x * x)));
}
__device__ __forceinline__ float gelu_grad(float x) {
  const float k0 = 0.7978845608028654f, k1 = 0.044715f;
  const float u = k0 * (x + k1 * x * x * x);
  const float th = tanhf(u);
  return 0.5f * (1.0f + th) + 0.5f * x * (1.0f - th * th) * k0 * (1.0f + 3.0f * k1 * x * x);
}

// ---------------------------------------------------------------- convolution (MFMA)
// out[s][p][co] = bias[co] + sum_{k, ci} w[co][k][ci] in[s][p + k - 2][ci]
// One workgroup per sample; wave v computes rows 32 (v & 1) .. +32 of output column
// tiles v / 2, v / 2 + 2, ...  mode 0: out_f32 = acc (+ bias), out_bf16 = bf16(that);
// mode 1: out_f32 = pre-activation, out_bf16 = bf16(gelu(pre)); mode 2: out_f32 += acc (+ bias).
template <int CIN, int TAPS>
__global__ void __launch_bounds__(256) conv_fwd_kernel(const uint16_t* __restrict__ in,
                                                       const uint16_t* __restrict__ w,
                                                       const float* __restrict__ bias, int cout, int dil, int mode,
                                                       float* __restrict__ out_f32, uint16_t* __restrict__ out_bf16) {
  constexpr int kStride = CIN + 4;  // padded LDS row: conflict-free 8-byte reads across a half wave
  __shared__ __align__(16) uint16_t xs[kPos * kStride];
  const int s = blockIdx.x;
  const int tid = threadIdx.x;
  const uint16_t* xin = in + static_cast<int64_t>(s) * kPos * CIN;
  for (int i = tid; i < kPos * CIN; i += 256) {
    const int row = i / CIN, c = i - row * CIN;
    xs[row * kStride + c] = xin[i];
  }
  __syncthreads();
  const int wave = tid >> 6, lane = tid & 63;
  const int half = wave & 1;
  const int m = lane & 31, kq = lane >> 5;
  for (int ct = wave >> 1; ct < cout / 32; ct += 2) {
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    const int co = ct * 32 + m;
    const uint16_t* wrow = w + static_cast<int64_t>(co) * TAPS * CIN + 4 * kq;
#pragma unroll
    for (int k = 0; k < TAPS; ++k) {
      const uint16_t* arow = xs + ((32 * half + m + (k - TAPS / 2) * dil) & (kPos - 1)) * kStride + 4 * kq;
#pragma unroll 4
      for (int c0 = 0; c0 < CIN; c0 += 8) {
        const bf16x4 a = *reinterpret_cast<const bf16x4*>(arow + c0);
        const bf16x4 b = *reinterpret_cast<const bf16x4*>(wrow + k * CIN + c0);
        acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, b, acc, 0, 0, 0);
      }
    }
    const float bv = bias ? bias[co] : 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int p = 32 * half + (r >> 2) * 8 + kq * 4 + (r & 3);
      const int64_t o = (static_cast<int64_t>(s) * kPos + p) * cout + co;
      const float v = acc[r] + bv;
      if (mode == 2) {
        out_f32[o] += v;
        continue;
      }
      if (out_f32) out_f32[o] = v;
      if (out_bf16) out_bf16[o] = f2bf(mode == 1 ? gelu(v) : v);
    }
  }
}

// ---------------------------------------------------------------- elementwise
__global__ void __launch_bounds__(256) gelu_bwd_kernel(const float* __restrict__ grad, const float* __restrict__ pre,
                                                       int64_t n, uint16_t* __restrict__ dz) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) dz[i] = f2bf(grad[i] * gelu_grad(pre[i]));
}

__global__ void __launch_bounds__(256) to_bf16_kernel(const float* __restrict__ x, int64_t n, uint16_t* __restrict__ y) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) y[i] = f2bf(x[i]);
}

// ---------------------------------------------------------------- weight gradient
// part[chunk][co][k][ci] = sum over the chunk's rows of dz[s][p][co] in[s][p + k - 2][ci]
// part_bias[chunk][co] = sum dz.  Workgroup: one chunk of samples x a 32 (co) x 64 (k, ci) tile.
constexpr int kWgSamples = 32;

__global__ void __launch_bounds__(256) wgrad_kernel(const uint16_t* __restrict__ dz, const uint16_t* __restrict__ in,
                                                    int num_samples, int cout, int cin, int taps, int dil,
                                                    float* __restrict__ part, float* __restrict__ part_bias) {
  __shared__ float dzs[kPos][33];
  __shared__ float xs[kPos][65];
  const int chunk = blockIdx.x;
  const int co0 = blockIdx.y * 32;
  const int kcols = taps * cin;
  const int halo = taps / 2;
  const int kc0 = blockIdx.z * 64;
  const int tid = threadIdx.x;
  // thread: co = co0 + (tid & 31), columns kc0 + (tid >> 5) + 8 j, j = 0..7
  const int tco = tid & 31, tcol = tid >> 5;
  float acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = 0.0f;
  float accb = 0.0f;
  const int s_end = std::min(num_samples, (chunk + 1) * kWgSamples);
  for (int s = chunk * kWgSamples; s < s_end; ++s) {
    for (int i = tid; i < kPos * 32; i += 256) {
      const int p = i >> 5, c = i & 31;
      dzs[p][c] = co0 + c < cout ? bf2f(dz[(static_cast<int64_t>(s) * kPos + p) * cout + co0 + c]) : 0.0f;
    }
    // input columns kc0 .. kc0 + 63 of the im2col row: (k, ci) = divmod(col, cin)
    for (int i = tid; i < kPos * 64; i += 256) {
      const int p = i >> 6, c = i & 63;
      const int col = kc0 + c;
      float v = 0.0f;
      if (col < kcols) {
        const int k = col / cin, ci = col - k * cin;
        const int q = (p + (k - halo) * dil) & (kPos - 1);  // input position feeding output p through tap k
        v = bf2f(in[(static_cast<int64_t>(s) * kPos + q) * cin + ci]);
      }
      xs[p][c] = v;
    }
    __syncthreads();
    for (int p = 0; p < kPos; ++p) {
      const float g = dzs[p][tco];
      if (tcol == 0) accb += g;
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] = fmaf(g, xs[p][tcol + 8 * j], acc[j]);
    }
    __syncthreads();
  }
  const int co = co0 + tco;
  if (co < cout) {
    float* prow = part + (static_cast<int64_t>(chunk) * cout + co) * kcols;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int col = kc0 + tcol + 8 * j;
      if (col < kcols) prow[col] = acc[j];
    }
    if (tcol == 0 && blockIdx.z == 0) part_bias[static_cast<int64_t>(chunk) * cout + co] = accb;
  }
}

// The same partial sums, bit for bit, on the float32 matrix cores.  A K = 1 MFMA adds one product to every
// accumulator with one rounding, so a chain of them over the chunk's positions is the chain of fmas above (a
// bf16 MFMA, nearly five times as fast here, sums 16 products in an order of its own; Adam carries that into the
// weights, activations round to other bfloat16 values, and the losses that follow leave the tenth digit).
// v_mfma_f32_16x16x1_4b makes four 16 x 16 blocks at once: a wavefront owns four blocks (16 output channels by 16
// (tap, ci) columns), the blocks of a workgroup's co group numbered channels first, so any four share an
// instruction and no shape pads more than its last one.  A workgroup holds one
// sample's dz columns and input rows in LDS (the next sample's are in flight in registers); memory holds
// channels innermost, so the operands come through the transposing LDS read, four positions of a lane's channel at a time
// (one read per position and operand took twice as long).  The input rows lie there twice, so that a tap's
// circular shift is a fixed distance from the position and all 64 steps read at constant offsets.  Each row ends
// in ones, the column of the bias gradient.
// Bound: float32 MFMA, 32 cycles a step and wavefront, and whole rounds of the 1024 SIMDs.  4096 samples on
// MI355X: 64 -> 224 channels 430 us, 8 -> 224 with 17 taps 177 us, 64 -> 64 133 us (the VALU kernel above: 1546, 931 and 457 us).
// Wavefronts of a workgroup: eight where its dz columns take most of the LDS, so that a CU holds 16 (64 -> 224, 4096
// samples: 430 us, with four 503), else four, which spread evenly over the CUs (64 -> 64: 133 us, with eight 164).
constexpr int wgrad_waves(int cot) { return cot > 2 ? 8 : 4; }

typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx2 __attribute__((ext_vector_type(2)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) shortx4 lds_shortx4;

// Row strides in elements: 32 bytes mod 128, so that the four rows of a transposing read lie on different banks.
constexpr int wgrad_dz_stride(int cot) { return cot * 32 + (cot % 2 == 0 ? 16 : 48); }
constexpr int kWgXStride = 64 + 16;  // (the ones behind the channels)

// Four rows of this lane's column of a 16-column tile per 16 lanes; `p`: the row (lane / 4) % 4 and the columns
// from 4 (lane % 4) of the tile that this lane names.
__device__ __forceinline__ uintx2 lds_read_tr(const uint16_t* p) {
  return __builtin_bit_cast(uintx2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4*)p));
}

// COT: 32-channel tiles of a workgroup's co group.
template <int COT>
__global__ void __launch_bounds__(64 * wgrad_waves(COT)) wgrad_mfma_kernel(const uint16_t* __restrict__ dz,
                                                                  const uint16_t* __restrict__ in, int num_samples,
                                                                  int cout, int cin, int taps, int dil,
                                                                  float* __restrict__ part,
                                                                  float* __restrict__ part_bias) {
  constexpr int DS = wgrad_dz_stride(COT);
  constexpr int kWaves = wgrad_waves(COT), kThreads = 64 * kWaves;
  constexpr int kDzVecs = kPos * COT * 32 / 8;  // 16-byte vectors of a sample's dz
  constexpr int kDzEach = (kDzVecs + kThreads - 1) / kThreads;
  constexpr int kXEach = kPos * 64 / 8 / kThreads;  // at most 64 input channels
  extern __shared__ __align__(16) uint16_t wg_lds[];
  uint16_t* dzs = wg_lds;
  uint16_t* xs = dzs + kPos * DS;
  constexpr int XS = kWgXStride;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int co0 = blockIdx.y * COT * 32;
  const int kcols = taps * cin;
  const int chunk = blockIdx.x;
  const int s_begin = chunk * kWgSamples;
  const int s_end = std::min(num_samples, s_begin + kWgSamples);
  // the rows and columns this lane names in the transposing reads of its block (channel and (tap, ci) tile); the
  // columns from kcols are ones: the bias column, and padding, which is dropped
  constexpr int kCoBlocks = 2 * COT;
  const int col_blocks = kcols / 16 + 1;
  const int first_block = 4 * (static_cast<int>(blockIdx.z) * kWaves + wave);
  const bool active = first_block < kCoBlocks * col_blocks;  // (whole wavefronts)
  const int block = std::min(first_block + (lane >> 4), kCoBlocks * col_blocks - 1);
  const int row4 = (lane >> 2) & 3;
  const int col = 16 * (block / kCoBlocks) + 4 * (lane & 3);
  const bool real = col < kcols;
  const int tap = real ? col / cin : 0;
  const uint16_t* az = dzs + row4 * DS + 16 * (block % kCoBlocks) + 4 * (lane & 3);
  const uint16_t* bx =
      xs + (row4 + (real ? ((tap - taps / 2) * dil) & (kPos - 1) : 0)) * XS + (real ? col - tap * cin : cin);
  for (int i = tid; i < 2 * kPos * 4; i += kThreads) xs[(i >> 2) * XS + cin + (i & 3)] = 0x3f80;  // bf16 1

  uintx4 rdz[kDzEach], rx[kXEach];
  const int xvecs = kPos * cin / 8;
  auto load = [&](int s) __attribute__((always_inline)) {
    const uint16_t* d = dz + static_cast<int64_t>(s) * kPos * cout + co0;
#pragma unroll
    for (int i = 0; i < kDzEach; ++i) {
      const int v = std::min(tid + i * kThreads, kDzVecs - 1);
      const int p = v / (COT * 4), c = v - p * (COT * 4);
      rdz[i] = *reinterpret_cast<const uintx4*>(d + p * cout + 8 * c);
    }
    const uintx4* x = reinterpret_cast<const uintx4*>(in + static_cast<int64_t>(s) * kPos * cin);
#pragma unroll
    for (int i = 0; i < kXEach; ++i) rx[i] = x[std::min(tid + i * kThreads, xvecs - 1)];
  };
  floatx16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  const int xrow_vecs = cin / 8;
  load(s_begin);
  for (int s = s_begin; s < s_end; ++s) {
#pragma unroll
    for (int i = 0; i < kDzEach; ++i) {
      const int v = tid + i * kThreads;
      const int p = v / (COT * 4), c = v - p * (COT * 4);
      if (v < kDzVecs) *reinterpret_cast<uintx4*>(dzs + p * DS + 8 * c) = rdz[i];
    }
#pragma unroll
    for (int i = 0; i < kXEach; ++i) {
      const int v = tid + i * kThreads;
      if (v < xvecs) {
        const int p = v / xrow_vecs, c = v - p * xrow_vecs;
        *reinterpret_cast<uintx4*>(xs + p * XS + 8 * c) = rx[i];
        *reinterpret_cast<uintx4*>(xs + (p + kPos) * XS + 8 * c) = rx[i];
      }
    }
    __syncthreads();
    if (s + 1 < s_end) load(s + 1);
    if (active) {
      // 16 positions' operands are read while those before them are multiplied
      constexpr int kReads = 4, kBatches = kPos / (4 * kReads);
      uintx2 a[2][kReads], b[2][kReads];
      auto read = [&](int q) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < kReads; ++j) {
          a[q & 1][j] = lds_read_tr(az + 4 * (kReads * q + j) * DS);
          b[q & 1][j] = lds_read_tr(bx + 4 * (kReads * q + j) * XS);
        }
      };
      auto value = [](uintx2 v, int i) __attribute__((always_inline)) {
        return __uint_as_float(i & 1 ? v[i >> 1] & 0xffff0000u : v[i >> 1] << 16);
      };
      read(0);
#pragma unroll
      for (int q = 0; q < kBatches; ++q) {
        if (q + 1 < kBatches) read(q + 1);
        __builtin_amdgcn_sched_barrier(0);  // (the compiler would read each operand where it is used)
#pragma unroll
        for (int j = 0; j < kReads; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            acc = __builtin_amdgcn_mfma_f32_16x16x1f32(value(a[q & 1][j], i), value(b[q & 1][j], i), acc, 0, 0, 0);
      }
    }
    __syncthreads();
  }
  if (!active) return;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int bl = first_block + b;
    if (bl >= kCoBlocks * col_blocks) break;
    const int oc = 16 * (bl / kCoBlocks) + (lane & 15);
    if (oc > kcols) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t row = static_cast<int64_t>(chunk) * cout + co0 + 16 * (bl % kCoBlocks) + 4 * (lane >> 4) + r;
      if (oc < kcols) part[row * kcols + oc] = acc[4 * b + r];
      else part_bias[row] = acc[4 * b + r];
    }
  }
}

// out[i] = sum of the chunks' partials of entry i in their order, weights then biases.  One thread per entry; 32
// chunks' values are read ahead of their additions, which are one chain (read one by one they were
// latency-bound: 31 us for 128 chunks of any size, 5 us now).
__global__ void __launch_bounds__(256) reduce_parts_kernel(const float* __restrict__ part_w, int64_t nw,
                                                           const float* __restrict__ part_b, int64_t nb, int chunks,
                                                           float* __restrict__ grad_w, float* __restrict__ grad_b) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= nw + nb) return;
  const bool weight = i < nw;
  const int64_t n = weight ? nw : nb;
  if (!weight) i -= nw;
  const float* part = (weight ? part_w : part_b) + i;
  constexpr int kAhead = 32;
  float s = 0.0f;
  int c = 0;
  for (; c + kAhead <= chunks; c += kAhead) {
    float v[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) v[j] = part[static_cast<int64_t>(c + j) * n];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) s += v[j];
  }
#pragma unroll 4
  for (; c < chunks; ++c) s += part[static_cast<int64_t>(c) * n];
  (weight ? grad_w : grad_b)[i] = s;
}

// ---------------------------------------------------------------- pilots in, grid out
// in[s][p][c]: c = 2 v + {0: re, 1: im} of LS value v * 64 + p (v = pilot word), c = 2 V: +-1 stream flag
// -log10(noise power) / 3: the SNR the receiver knows (0 dB -> 0, 30 dB -> 1 at unit signal power)
__device__ __forceinline__ float snr_feature(const double* noise_power, int64_t d) {
  return noise_power ? static_cast<float>(-log10(noise_power[d]) / 3.0) : 0.0f;
}

__global__ void __launch_bounds__(256) net_input_kernel(const float2* __restrict__ ls, int64_t num_samples,
                                                        int num_drops, int num_rx, int pilot_words, int cin,
                                                        const double* __restrict__ noise_power,
                                                        uint16_t* __restrict__ x) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= num_samples * kPos) return;
  const int64_t s = i / kPos;
  const int p = static_cast<int>(i - s * kPos);
  const int t = static_cast<int>(s / (static_cast<int64_t>(num_drops) * num_rx));
  const float2* row = ls + s * pilot_words * kPos;
  uint16_t* o = x + i * cin;
  for (int v = 0; v < pilot_words; ++v) {
    const float2 h = row[v * kPos + p];
    o[2 * v] = f2bf(h.x);
    o[2 * v + 1] = f2bf(h.y);
  }
  o[2 * pilot_words] = f2bf(t ? 1.0f : -1.0f);
  o[2 * pilot_words + 1] = f2bf(snr_feature(noise_power, (s % (static_cast<int64_t>(num_drops) * num_rx)) / num_rx));
  for (int c = 2 * pilot_words + 2; c < cin; ++c) o[c] = 0;
}

// out[s][p][c], c = (w * B + u) * 2 + {re, im} -> est[s][w][B p + u]  (B = N / 64 subcarriers per position)
__global__ void __launch_bounds__(256) net_output_kernel(const float* __restrict__ out, int64_t num_samples, int words,
                                                         int n, float2* __restrict__ est) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t wn = static_cast<int64_t>(words) * n;
  if (i >= num_samples * wn) return;
  const int64_t s = i / wn;
  const int e = static_cast<int>(i - s * wn);
  const int w = e / n, q = e - w * n;
  const int blk = n / kPos;
  const int p = q / blk, u = q - p * blk;
  const int cout = 2 * words * blk;
  const float* o = out + (s * kPos + p) * cout + 2 * (w * blk + u);
  est[i] = make_float2(o[0], o[1]);
}

// ---------------------------------------------------------------- NMSE against the ideal CSI
// H[s][w][q] = S[d][r][t] c[d][w][q];  acc[0] += |est - H|^2, acc[1] += |H|^2 (per drop when per_drop)
__device__ __forceinline__ float2 ideal_h(const float2* csi, const float2* spatial, int64_t s, int64_t e, int num_drops,
                                          int num_rx, int num_tx, int64_t wn) {
  const int64_t dr = s % (static_cast<int64_t>(num_drops) * num_rx);
  const int t = static_cast<int>(s / (static_cast<int64_t>(num_drops) * num_rx));
  const int64_t d = dr / num_rx;
  const int r = static_cast<int>(dr - d * num_rx);
  return cmul(spatial[(d * num_rx + r) * num_tx + t], csi[d * wn + e]);
}

// the same factor by factor: the sample's entry of S and its drop's csi
__device__ __forceinline__ const float2* ideal_parts(const float2* csi, const float2* spatial, int64_t s, int num_drops,
                                                     int num_rx, int num_tx, int64_t wn, float2* sp) {
  const int64_t dr = s % (static_cast<int64_t>(num_drops) * num_rx);
  const int t = static_cast<int>(s / (static_cast<int64_t>(num_drops) * num_rx));
  const int64_t d = dr / num_rx;
  const int r = static_cast<int>(dr - d * num_rx);
  *sp = spatial[(d * num_rx + r) * num_tx + t];
  return csi + d * wn;
}

__global__ void __launch_bounds__(256) estimate_error_kernel(const float2* __restrict__ est,
                                                             const float2* __restrict__ csi,
                                                             const float2* __restrict__ spatial, int num_drops,
                                                             int num_rx, int num_tx, int64_t wn,
                                                             double* __restrict__ err, double* __restrict__ pow) {
  // one workgroup per (sample); per-drop sums
  __shared__ double red[2][4];
  const int64_t s = blockIdx.x;
  double e2 = 0.0, h2 = 0.0;
  for (int64_t e = threadIdx.x; e < wn; e += blockDim.x) {
    const float2 h = ideal_h(csi, spatial, s, e, num_drops, num_rx, num_tx, wn);
    const float2 x = est[s * wn + e];
    e2 += static_cast<double>(cabs2(csub(x, h)));
    h2 += static_cast<double>(cabs2(h));
  }
  for (int off = 32; off > 0; off >>= 1) {
    e2 += __shfl_down(e2, off, 64);
    h2 += __shfl_down(h2, off, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = e2;
    red[1][threadIdx.x >> 6] = h2;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int64_t d = (s % (static_cast<int64_t>(num_drops) * num_rx)) / num_rx;
    atomicAdd(err + d, red[0][0] + red[0][1] + red[0][2] + red[0][3]);
    atomicAdd(pow + d, red[1][0] + red[1][1] + red[1][2] + red[1][3]);
  }
}

// Loss of a batch: mean over SNR groups of the NMSE in dB, 10 log10(sum |out - H|^2 / sum |H|^2) per
// group, so that every SNR point weighs alike (a batch NMSE would be dominated by the noisiest
// drops).  Pass 1 accumulates per-group error and power (one workgroup per sample), pass 2 turns
// them into the loss and per-group gradient scales, pass 3 writes d loss / d out.
__device__ __forceinline__ int64_t out_index(int64_t s, int e, int words, int n) {
  const int w = e / n, q = e - w * n;
  const int blk = n / kPos;
  const int p = q / blk, u = q - p * blk;
  return (s * kPos + p) * (2 * words * blk) + 2 * (w * blk + u);
}

// The gradient pass walks a sample's output as it lies in memory, one (re, im) pair per thread and step.
// Threads 256 apart differ by a fixed (position, word, subcarrier) step, so the pair's place is carried along
// instead of divided out each time, and reads of the output and writes of the gradient are whole lines:
// 4096 samples of 224 channels 90 us, bfloat16 gradients (159 us, and 117 us for the conversion, before).
// (The accumulation keeps the grid's order and so the order of its sums: 128 us, 129 in this one.)
struct PairWalk {
  int p, w, u;  // position, word, subcarrier of the position: subcarrier blk p + u of word w
  int dp, dw, du, blk, words;
  __device__ __forceinline__ PairWalk(int first, int step, int words_, int n) : blk(n / kPos), words(words_) {
    const int per = words * blk;
    p = first / per;
    w = (first - p * per) / blk;
    u = first - p * per - w * blk;
    dp = step / per;
    dw = (step - dp * per) / blk;
    du = step - dp * per - dw * blk;
  }
  __device__ __forceinline__ void next() {
    u += du;
    w += dw;
    p += dp;
    if (u >= blk) {
      u -= blk;
      ++w;
    }
    if (w >= words) {
      w -= words;
      ++p;
    }
  }
  __device__ __forceinline__ int element(int n) const { return w * n + blk * p + u; }
};

__device__ __forceinline__ int sample_group(int64_t s, int num_drops, int num_rx, const int32_t* group) {
  const int64_t d = (s % (static_cast<int64_t>(num_drops) * num_rx)) / num_rx;
  return group ? group[d] : 0;
}

__global__ void __launch_bounds__(256) loss_accumulate_kernel(const float* __restrict__ out,
                                                              const float2* __restrict__ csi,
                                                              const float2* __restrict__ spatial, int num_drops,
                                                              int num_rx, int num_tx, int words, int n,
                                                              const int32_t* __restrict__ group, int num_groups,
                                                              double* __restrict__ work) {
  __shared__ double red[2][4];
  const int64_t s = blockIdx.x;
  const int64_t wn = static_cast<int64_t>(words) * n;
  double e2 = 0.0, h2 = 0.0;
  for (int e = threadIdx.x; e < wn; e += blockDim.x) {
    const float2 h = ideal_h(csi, spatial, s, e, num_drops, num_rx, num_tx, wn);
    const int64_t o = out_index(s, e, words, n);
    const float dr = out[o] - h.x, di = out[o + 1] - h.y;
    e2 += static_cast<double>(dr * dr + di * di);
    h2 += static_cast<double>(cabs2(h));
  }
  for (int off = 32; off > 0; off >>= 1) {
    e2 += __shfl_down(e2, off, 64);
    h2 += __shfl_down(h2, off, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = e2;
    red[1][threadIdx.x >> 6] = h2;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int g = sample_group(s, num_drops, num_rx, group);
    atomicAdd(work + g, red[0][0] + red[0][1] + red[0][2] + red[0][3]);
    atomicAdd(work + num_groups + g, red[1][0] + red[1][1] + red[1][2] + red[1][3]);
  }
}

__global__ void loss_finish_kernel(int num_groups, double* __restrict__ work, double* __restrict__ loss) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  double l = 0.0;
  int used = 0;
  for (int g = 0; g < num_groups; ++g) {
    const double err = work[g], pw = work[num_groups + g];
    if (err > 0.0 && pw > 0.0) {
      l += 10.0 * log10(err / pw);
      ++used;
    }
  }
  // d/d out of mean_g 10 log10(err_g / pow_g) = (10 / ln 10) / (used err_g) * 2 (out - H)
  for (int g = 0; g < num_groups; ++g)
    work[2 * num_groups + g] = (work[g] > 0.0 && used) ? 2.0 * 4.342944819032518 / (used * work[g]) : 0.0;
  loss[0] = used ? l / used : 0.0;
}

// Workgroup (sample, share of its pairs); GRAD: float, or bfloat16 (uint16_t) for the backward pass.
template <class GRAD>
__global__ void __launch_bounds__(256) loss_grad_kernel(const float* __restrict__ out, const float2* __restrict__ csi,
                                                        const float2* __restrict__ spatial, int num_drops, int num_rx,
                                                        int num_tx, int words, int n, const int32_t* __restrict__ group,
                                                        int num_groups, const double* __restrict__ work,
                                                        GRAD* __restrict__ grad) {
  const int64_t s = blockIdx.x;
  const int64_t wn = static_cast<int64_t>(words) * n;
  const float* row = out + 2 * s * wn;  // (aligned as floats are, like the gradient)
  float2 sp;
  const float2* c = ideal_parts(csi, spatial, s, num_drops, num_rx, num_tx, wn, &sp);
  const float scale = static_cast<float>(work[2 * num_groups + sample_group(s, num_drops, num_rx, group)]);
  const int first = static_cast<int>(blockIdx.y * blockDim.x + threadIdx.x);
  const int step = static_cast<int>(gridDim.y * blockDim.x);
  PairWalk at(first, step, words, n);
#pragma unroll 4
  for (int i = first; i < wn; i += step, at.next()) {
    const float2 h = cmul(sp, c[at.element(n)]);
    float v[2];
    __builtin_memcpy(v, row + 2 * i, sizeof(v));
    const float gr = scale * (v[0] - h.x), gi = scale * (v[1] - h.y);
    GRAD pair[2];
    if constexpr (sizeof(GRAD) == 2) {
      pair[0] = f2bf(gr);
      pair[1] = f2bf(gi);
    } else {
      pair[0] = gr;
      pair[1] = gi;
    }
    __builtin_memcpy(grad + 2 * (s * wn + i), pair, sizeof(pair));
  }
}

// ---------------------------------------------------------------- Adam + weight copies
// params float32 [cout][5][cin] (+ bias [cout] separately); writes w_bf16 [cout][5][cin] and the
// transposed, flipped copy wt_bf16 [cin][5][cout] (wt[ci][k][co] = w[co][4 - k][ci]) used by
// the backward-data convolution.
__device__ __forceinline__ float adam_update(float* p, const float* g, float* m1, float* m2, int64_t i, float lr,
                                             float b1, float b2, float eps, float c1, float c2) {
  const float gi = g[i];
  const float a = b1 * m1[i] + (1.0f - b1) * gi;
  const float b = b2 * m2[i] + (1.0f - b2) * gi * gi;
  m1[i] = a;
  m2[i] = b;
  const float v = p[i] - lr * (a / c1) / (sqrtf(b / c2) + eps);
  p[i] = v;
  return v;
}

__global__ void __launch_bounds__(256) adam_kernel(float* __restrict__ p, const float* __restrict__ g,
                                                   float* __restrict__ m1, float* __restrict__ m2, int64_t n, float lr,
                                                   float b1, float b2, float eps, float c1, float c2) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) adam_update(p, g, m1, m2, i, lr, b1, b2, eps, c1, c2);
}

// Every parameter tensor of a network in one launch, the weights' bfloat16 copies with them (ten updates and
// five copies of at most 72 K elements were 15 launches of 4.5 us each).
struct AdamTensors {
  hpx_adam_tensor t[HPX_ADAM_MAX_TENSORS];
  int first_block[HPX_ADAM_MAX_TENSORS + 1];
  int count;
};

__global__ void __launch_bounds__(256) adam_tensors_kernel(AdamTensors a, float lr, float b1, float b2, float eps,
                                                           float c1, float c2) {
  int k = 0;
  while (k + 1 < a.count && static_cast<int>(blockIdx.x) >= a.first_block[k + 1]) ++k;
  const hpx_adam_tensor& t = a.t[k];
  const int64_t i = static_cast<int64_t>(static_cast<int>(blockIdx.x) - a.first_block[k]) * 256 + threadIdx.x;
  if (i >= t.n) return;
  const uint16_t v = f2bf(adam_update(t.param, t.grad, t.m1, t.m2, i, lr, b1, b2, eps, c1, c2));
  if (t.weight) t.weight[i] = v;
  if (t.weight_transposed) {
    const int row = t.taps * t.cin;
    const int co = static_cast<int>(i / row), rest = static_cast<int>(i - static_cast<int64_t>(co) * row);
    const int tap = rest / t.cin, ci = rest - tap * t.cin;
    t.weight_transposed[(static_cast<int64_t>(ci) * t.taps + (t.taps - 1 - tap)) * (t.n / row) + co] = v;
  }
}

__global__ void __launch_bounds__(256) weight_copies_kernel(const float* __restrict__ p, int cout, int cin, int taps,
                                                            uint16_t* __restrict__ w, uint16_t* __restrict__ wt) {
  const int64_t n = static_cast<int64_t>(cout) * taps * cin;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int co = static_cast<int>(i / (taps * cin));
  const int rest = static_cast<int>(i - static_cast<int64_t>(co) * taps * cin);
  const int k = rest / cin, ci = rest - k * cin;
  const uint16_t v = f2bf(p[i]);
  if (w) w[i] = v;
  if (wt) wt[(static_cast<int64_t>(ci) * taps + (taps - 1 - k)) * cout + co] = v;
}

// ---------------------------------------------------------------- fused passes over the network
// A workgroup of four wavefronts takes 2 PT samples through the whole network with every activation in
// LDS; a wavefront owns PT tiles of 32 positions and computes all output channels of them.  Weights
// are the A operand of the 32x32x16 bf16 MFMA and activations the B operand, so a lane ends up
// with four consecutive channels of one position: activations go back to LDS, and results to memory,
// as whole 8- and 16-byte pieces.  Two channel tiles are computed together, so that one activation
// read feeds two MFMAs and one weight read PT of them (one tile a wavefront and four samples read
// 1 KB of LDS per MFMA, which is all the LDS bandwidth there is).  A layer is computed in place: its
// input is read in full into accumulators before its output is written, and with PT >= 2 a
// wavefront owns whole samples.  Rows of 64 channels are stored with their 16-byte pieces permuted by
// row (piece ^ (row & 7)), free of bank conflicts without padding: 44 KB for four samples, three workgroups
// per CU.  All sums keep the order of the layer-by-layer convolutions and so round to the same bfloat16.
// 16384 samples of 224 output channels on MI355X: 647 -> 484 us (630 TFLOP/s; the VALU, with tanhf 28 of
// some 33 instructions per hidden value, is busy for 65 % of it and the matrix cores for 31 %); eight
// samples a workgroup 495 us, one sample two wavefronts 527 us.
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4n __attribute__((ext_vector_type(4)));
constexpr int kActElems = kPos * 64;  // a sample's activations

struct NetWeights {
  const uint16_t* w[5];  // bfloat16 [cout][taps][cin]: four layers, skip
  const float* b[5];
};

// This lane's place in the 32x32 tiles: column (position) m, half kq of the contraction / of the rows.
struct TileLane {
  int wave, m, kq;
  __device__ __forceinline__ TileLane()
      : wave(static_cast<int>(threadIdx.x) >> 6), m(static_cast<int>(threadIdx.x) & 31), kq((static_cast<int>(threadIdx.x) >> 5) & 1) {}
  // tile t of the wavefront's PT: sample of the group and half of its positions
  template <int PT>
  __device__ __forceinline__ int sample(int t) const { return (wave * PT + t) >> 1; }
  template <int PT>
  __device__ __forceinline__ int half(int t) const { return PT == 1 ? wave & 1 : t & 1; }
};

// Orders LDS accesses of the lanes that share a sample.
template <int PT>
__device__ __forceinline__ void sample_sync() {
  if constexpr (PT == 1) {
    __syncthreads();
  } else {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

template <int PT, int CT>
__device__ __forceinline__ void zero_tiles(floatx16 (&acc)[CT][PT]) {
#pragma unroll
  for (int c = 0; c < CT; ++c)
#pragma unroll
    for (int t = 0; t < PT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[c][t][r] = 0.0f;
}

// Eight weights in one load, wherever they lie: the caller's weights need no more than their own alignment.
__device__ __forceinline__ uintx4 load8(const uint16_t* p) {
  uintx4 v;
  __builtin_memcpy(&v, p, sizeof(v));
  return v;
}

// Weights on their way to LDS: the workgroup loads a chunk (up to 64 output channels by 64 elements of
// their rows, whole 128-byte lines) into registers while the chunk before it is in use, and all
// wavefronts read their fragments from the copy in LDS, rows permuted like the activations'.  (Fragments
// read by each wavefront from memory touch 32 lines for 1 KB: 16384 samples, eight a workgroup, 536 us so, 495 us
// through LDS.)
struct WeightPipe {
  uint16_t* lds;
  uintx4 r0, r1;
  // rows of 16 STEPS elements
  template <int ROWS, int STEPS>
  __device__ __forceinline__ void fetch(const uint16_t* __restrict__ w, int64_t wrow) {
    constexpr int kPieces = 2 * STEPS, kTotal = ROWS * kPieces;
    static_assert(kTotal == 256 || kTotal == 512, "one or two whole pieces per thread");
    const int row = static_cast<int>(threadIdx.x) / kPieces, c = static_cast<int>(threadIdx.x) % kPieces;
    const uint16_t* p = w + row * wrow + 8 * c;
    r0 = load8(p);
    if constexpr (kTotal == 512) r1 = load8(p + (256 / kPieces) * wrow);
  }
  template <int ROWS, int STEPS>
  __device__ __forceinline__ void commit() {
    constexpr int kPieces = 2 * STEPS, kTotal = ROWS * kPieces;
    const int row = static_cast<int>(threadIdx.x) / kPieces, c = static_cast<int>(threadIdx.x) % kPieces;
    uint16_t* p = lds + (row << 6) + ((c ^ (row & 7)) << 3);
    __syncthreads();  // the chunk before is read
    *reinterpret_cast<uintx4*>(p) = r0;
    if constexpr (kTotal == 512) *reinterpret_cast<uintx4*>(p + (256 / kPieces) * 64) = r1;
    __syncthreads();
  }
  __device__ __forceinline__ bf16x8 fragment(int tile, int step, const TileLane& ln) const {
    return *reinterpret_cast<const bf16x8*>(lds + ((32 * tile + ln.m) << 6) + (((2 * step + ln.kq) ^ (ln.m & 7)) << 3));
  }
};

// acc += circular convolution of 16 STEPS input channels (w: the first tile's weights of these channels,
// rows of `wrow` elements, taps `wtap` apart).  Its first chunk is in the pipe already; `next` fetches
// the one that follows the last.
template <int PT, int CT, int STEPS, class Next>
__device__ __forceinline__ void conv_channels(const uint16_t* act, WeightPipe& pipe, const uint16_t* __restrict__ w, int64_t wrow,
                                              int wtap, int dil, const TileLane& ln, floatx16 (&acc)[CT][PT], Next next) {
#pragma unroll 1
  for (int k = 0; k < kTaps; ++k) {
    pipe.template commit<32 * CT, STEPS>();
    if (k + 1 < kTaps) pipe.template fetch<32 * CT, STEPS>(w + (k + 1) * wtap, wrow);
    else next();
    const int row = (ln.m + (k - kTaps / 2) * dil) & (kPos - 1);  // (the other half of the positions: row ^ 32)
    const int sw = row & 7;
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
      const int piece = ((2 * j + ln.kq) ^ sw) << 3;
      bf16x8 wv[CT];
#pragma unroll
      for (int c = 0; c < CT; ++c) wv[c] = pipe.fragment(c, j, ln);
#pragma unroll
      for (int t = 0; t < PT; ++t) {
        const uint16_t* a = act + ln.template sample<PT>(t) * kActElems + ((row ^ (32 * ln.template half<PT>(t))) << 6) + piece;
        const bf16x8 v = *reinterpret_cast<const bf16x8*>(a);
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[c][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv[c], v, acc[c][t], 0, 0, 0);
      }
    }
  }
}

// The same from the 8-channel input rows: a step takes two taps (lanes 0-31 the even one, 32-63 the odd
// one; the tap beyond the last has zero weights).  These weights come straight from memory (9 KB a tile).
template <int PT, int CT, int TAPS>
__device__ __forceinline__ void conv_input(const uint16_t* xs, const uint16_t* __restrict__ w, const TileLane& ln,
                                           floatx16 (&acc)[CT][PT]) {
  const uint16_t* wl = w + ln.m * (TAPS * 8);
#pragma unroll 3
  for (int j = 0; j < (TAPS + 1) / 2; ++j) {
    const int tap = 2 * j + ln.kq;
    bf16x8 wv[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      uintx4 v = load8(wl + c * 32 * (TAPS * 8) + min(tap, TAPS - 1) * 8);
      if (tap >= TAPS) v = uintx4{0u, 0u, 0u, 0u};
      wv[c] = __builtin_bit_cast(bf16x8, v);
    }
    const int row = (ln.m + tap - TAPS / 2) & (kPos - 1);
#pragma unroll
    for (int t = 0; t < PT; ++t) {
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(
          xs + (ln.template sample<PT>(t) * kPos + (row ^ (32 * ln.template half<PT>(t)))) * 8);
#pragma unroll
      for (int c = 0; c < CT; ++c) acc[c][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv[c], v, acc[c][t], 0, 0, 0);
    }
  }
}

// f(tile t, position, first of four channels, their values) over this lane's accumulators of channel tile c
template <int PT, int CT, class F>
__device__ __forceinline__ void each_quad(const floatx16 (&acc)[CT][PT], const TileLane& ln, F f) {
#pragma unroll
  for (int c = 0; c < CT; ++c)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int t = 0; t < PT; ++t)
        f(t, 32 * ln.template half<PT>(t) + ln.m, 32 * c + 8 * j + 4 * ln.kq,
          floatx4{acc[c][t][4 * j], acc[c][t][4 * j + 1], acc[c][t][4 * j + 2], acc[c][t][4 * j + 3]});
}

__device__ __forceinline__ floatx4 load4(const float* p) {
  floatx4 v;
  __builtin_memcpy(&v, p, sizeof(v));
  return v;
}

// where channels co .. co + 3 of position p lie in a sample's permuted rows
__device__ __forceinline__ int act_at(int p, int co) { return (p << 6) + (((co >> 3) ^ (p & 7)) << 3) + (co & 4); }

// What a training step keeps of the forward pass: per hidden layer the pre-activations and the
// activations (rows [sample][position][channel]), and the output.
struct Kept {
  float* pre[3];
  uint16_t* act[3];
  float* out;
};

// TRAIN: the input rows come from x and everything the backward pass needs goes to `kept`; otherwise
// the least-squares values of the sample's pilots come from the received grid and the estimate goes
// straight to its grid (VEC: four channels are two whole subcarriers of one word, 16-byte aligned).
template <int PT, bool TRAIN, bool VEC>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(PT == 1 ? 4 : 3)))
net_forward_kernel(const float2* __restrict__ grid, int num_drops, int num_rx, int words, int n,
                   const int32_t* __restrict__ pidx, const float2* __restrict__ pval, int num_pilots,
                   const double* __restrict__ noise_power, const uint16_t* __restrict__ x, int64_t num_samples,
                   NetWeights net, int cout, float* __restrict__ est, Kept kept) {
  constexpr int kGroup = 2 * PT;
  __shared__ __align__(16) uint16_t act[kGroup * kActElems];
  __shared__ __align__(16) uint16_t xs[kGroup * kPos * 8];
  __shared__ __align__(16) uint16_t chunk[64 * 64];
  WeightPipe pipe{chunk, uintx4{}, uintx4{}};
  pipe.fetch<64, 4>(net.w[1], kTaps * 64);
  const int tid = threadIdx.x;
  const int64_t s0 = static_cast<int64_t>(blockIdx.x) * kGroup;
  const int64_t wn = static_cast<int64_t>(words) * n;
  for (int i = tid; i < kGroup * kPos; i += 256) {
    const int g = i / kPos, p = i - g * kPos;
    const int64_t s = s0 + g;
    uintx4 row = uintx4{0u, 0u, 0u, 0u};
    if (s < num_samples) {
      if constexpr (TRAIN) {
        row = *reinterpret_cast<const uintx4*>(x + (s * kPos + p) * 8);
      } else {
        // LS at the sample's own pilots, two channels per pilot word, the stream flag, the SNR
        const int64_t dr_count = static_cast<int64_t>(num_drops) * num_rx;
        const int pilot_words = num_pilots / kPos;
        const int t = static_cast<int>(s / dr_count);
        const int64_t dr = s - t * dr_count;
        uint32_t pair[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int v = 0; v < 3; ++v) {
          if (v >= pilot_words) break;
          const int j = v * kPos + p;
          const float2 px = pval[t * num_pilots + j];
          const float2 y = grid[dr * wn + pidx[t * num_pilots + j]];
          // (the products in this order: the value decides which bfloat16 neighbour it rounds to)
          const float2 c = make_float2(fmaf(px.x, y.x, px.y * y.y), fmaf(-px.y, y.x, px.x * y.y));
          const float2 h = cscale(c, 1.0f / cabs2(px));
          pair[v] = f2bf(h.x) | static_cast<uint32_t>(f2bf(h.y)) << 16;
        }
        const uint32_t last = f2bf(t ? 1.0f : -1.0f) | static_cast<uint32_t>(f2bf(snr_feature(noise_power, dr / num_rx))) << 16;
#pragma unroll
        for (int v = 0; v < 4; ++v) row[v] = v == pilot_words ? last : pair[v];
      }
    }
    *reinterpret_cast<uintx4*>(xs + i * 8) = row;
  }
  __syncthreads();
  const TileLane ln;
  auto hidden = [&](int layer, const floatx16 (&acc)[2][PT]) __attribute__((always_inline)) {
    each_quad<PT, 2>(acc, ln, [&](int t, int p, int co, floatx4 v) __attribute__((always_inline)) {
      v += load4(net.b[layer] + co);
      bf16x4n h;
#pragma unroll
      for (int i = 0; i < 4; ++i) h[i] = static_cast<__bf16>(gelu(v[i]));
      const int g = ln.template sample<PT>(t);
      *reinterpret_cast<bf16x4n*>(act + g * kActElems + act_at(p, co)) = h;
      if constexpr (TRAIN) {
        if (s0 + g < num_samples) {
          const int64_t o = ((s0 + g) * kPos + p) * 64 + co;
          *reinterpret_cast<floatx4*>(kept.pre[layer] + o) = v;
        }
      }
    });
    sample_sync<PT>();
    // the activations from LDS, in whole lines (eight bytes a lane from the accumulators touch 32 lines a store)
    if constexpr (TRAIN) {
      constexpr int kLanes = 128;  // a sample's two wavefronts
      static_assert(PT == 1, "");
      const int g = ln.template sample<PT>(0);
      if (s0 + g < num_samples) {
        uint16_t* dst = kept.act[layer] + (s0 + g) * kActElems;
#pragma unroll
        for (int i = tid & (kLanes - 1); i < kActElems / 8; i += kLanes)
          *reinterpret_cast<uintx4*>(dst + 8 * i) =
              *reinterpret_cast<const uintx4*>(act + g * kActElems + act_at(i >> 3, 8 * (i & 7)));
      }
    }
  };
  {
    floatx16 acc[2][PT];
    zero_tiles<PT, 2>(acc);
    static_assert(kDil1 == 1, "");
    conv_input<PT, 2, kTaps>(xs, net.w[0], ln, acc);
    hidden(0, acc);
    zero_tiles<PT, 2>(acc);
    conv_channels<PT, 2, 4>(act, pipe, net.w[1], kTaps * 64, 64, kDil2, ln, acc,
                            [&]() __attribute__((always_inline)) { pipe.fetch<64, 4>(net.w[2], kTaps * 64); });
    sample_sync<PT>();
    hidden(1, acc);
    zero_tiles<PT, 2>(acc);
    conv_channels<PT, 2, 4>(act, pipe, net.w[2], kTaps * 64, 64, kDil3, ln, acc, [&]() __attribute__((always_inline)) {
      if (cout >= 64) pipe.fetch<64, 4>(net.w[3], kTaps * 64);
      else pipe.fetch<32, 4>(net.w[3], kTaps * 64);
    });
    sample_sync<PT>();
    hidden(2, acc);
  }
  // last layer, and the skip convolution a channel tile at a time
  const int blk = n / kPos;
  auto last = [&](auto tiles, int ct) __attribute__((always_inline)) {
    constexpr int CT = decltype(tiles)::value;
    floatx16 acc[CT][PT];
    zero_tiles<PT, CT>(acc);
    const uint16_t* w4 = net.w[3] + static_cast<int64_t>(ct) * 32 * kTaps * 64;
    conv_channels<PT, CT, 4>(act, pipe, w4, kTaps * 64, 64, kDil4, ln, acc, [&]() __attribute__((always_inline)) {  // (then the next tiles, if there are any)
      const uint16_t* after = w4 + 32 * CT * kTaps * 64;
      if (ct + CT + 1 < cout / 32) pipe.fetch<64, 4>(after, kTaps * 64);
      else if (ct + CT < cout / 32) pipe.fetch<32, 4>(after, kTaps * 64);
    });
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      floatx16 sk[1][PT];
      zero_tiles<PT, 1>(sk);
      conv_input<PT, 1, kSkipTaps>(xs, net.w[4] + static_cast<int64_t>(ct + c) * 32 * kSkipTaps * 8, ln, sk);
      each_quad<PT, 1>(sk, ln, [&](int t, int p, int cc, floatx4 skip) __attribute__((always_inline)) {
        const int64_t s = s0 + ln.template sample<PT>(t);
        const int co = 32 * (ct + c) + cc, j = (cc >> 3);
        const floatx4 main = floatx4{acc[c][t][4 * j], acc[c][t][4 * j + 1], acc[c][t][4 * j + 2], acc[c][t][4 * j + 3]};
        const floatx4 v = (main + load4(net.b[3] + co)) + (skip + load4(net.b[4] + co));
        if (s >= num_samples) return;
        if constexpr (TRAIN) {
          *reinterpret_cast<floatx4*>(kept.out + (s * kPos + p) * cout + co) = v;
        } else {
          // channel 2 (w B + u) + {re, im} of position p -> est[s][w][B p + u]
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int c2 = (co >> 1) + h;
            const int w = c2 / blk, u = c2 - w * blk;
            float* e = est + 2 * (s * wn + static_cast<int64_t>(w) * n + blk * p + u);
            if constexpr (VEC) {
              *reinterpret_cast<floatx4*>(e) = v;
              break;
            } else {
              *reinterpret_cast<float2*>(e) = make_float2(v[2 * h], v[2 * h + 1]);
            }
          }
        }
      });
    }
  };
  int ct = 0;
#pragma unroll 1
  for (; ct + 1 < cout / 32; ct += 2) last(std::integral_constant<int, 2>{}, ct);
  if (ct < cout / 32) last(std::integral_constant<int, 1>{}, ct);
}

// Backward through the data: dz of the output rows [sample][position][COUT] -> dz of the three hidden
// layers' pre-activations, each the transposed convolution (flipped weights [cin][taps][cout]) times
// GELU's derivative, rounded to bfloat16 for the next one and for the weight gradients.  The sums run
// over taps, then channels, as the layer-by-layer convolutions' do, so every value is theirs: the output
// rows of a sample lie in LDS whole (16 bytes behind each row: free of bank conflicts), which at 224 channels leaves
// room for two samples a workgroup and two workgroups a CU.  COUT: 224 and 64, the widths that the layer-by-layer
// backward convolution has (frames of 7168 and of 2048 elements).
struct Gradients {
  const uint16_t* wt[3];  // transposed weights of layers 2, 3, 4
  const float* pre[3];
  uint16_t* dz[3];
};

template <int COUT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
net_backward_kernel(const uint16_t* __restrict__ dz_out, int64_t num_samples, Gradients net) {
  constexpr int kGroup = 2, kOutRow = COUT + 8, kFull = COUT / 64;
  constexpr bool kHalf = COUT % 64 == 32;
  static_assert(kHalf || COUT % 64 == 0, "whole chunks, and at most a half one");
  __shared__ __align__(16) uint16_t rows[kGroup * kPos * kOutRow];
  __shared__ __align__(16) uint16_t chunk[64 * 64];
  uint16_t* act = rows;  // the hidden rows take the output rows' place
  WeightPipe pipe{chunk, uintx4{}, uintx4{}};
  constexpr int64_t wrow = kTaps * COUT;
  pipe.fetch<64, 4>(net.wt[2], wrow);
  const int64_t s0 = static_cast<int64_t>(blockIdx.x) * kGroup;
  constexpr int kPieces = COUT / 8;
#pragma unroll 7
  for (int i = threadIdx.x; i < kGroup * kPos * kPieces; i += 256) {
    const int row = i / kPieces, c = i - row * kPieces;  // (row: sample and position)
    const int64_t s = min(s0 + (row >> 6), num_samples - 1);
    *reinterpret_cast<uintx4*>(rows + row * kOutRow + 8 * c) =
        *reinterpret_cast<const uintx4*>(dz_out + (s * kPos + (row & 63)) * COUT + 8 * c);
  }
  const TileLane ln;
  const int g = ln.sample<1>(0), half = ln.half<1>(0);
  floatx16 acc[2][1];
  zero_tiles<1, 2>(acc);
  auto steps = [&](const uint16_t* a, auto count) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < decltype(count)::value; ++j) {
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(a + 16 * j);
#pragma unroll
      for (int c = 0; c < 2; ++c)
        acc[c][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pipe.fragment(c, j, ln), v, acc[c][0], 0, 0, 0);
    }
  };
#pragma unroll 1
  for (int k = 0; k < kTaps; ++k) {
    const uint16_t* w = net.wt[2] + k * COUT;
    const int row = ((ln.m + (k - kTaps / 2) * kDil4) & (kPos - 1)) ^ (32 * half);
    const uint16_t* a = rows + (g * kPos + row) * kOutRow + 8 * ln.kq;
    auto next_tap = [&]() __attribute__((always_inline)) {
      if (k + 1 < kTaps) pipe.fetch<64, 4>(w + COUT, wrow);
      else pipe.fetch<64, 4>(net.wt[1], kTaps * 64);
    };
#pragma unroll
    for (int q = 0; q < kFull; ++q) {
      pipe.commit<64, 4>();
      if (q + 1 < kFull) pipe.fetch<64, 4>(w + 64 * (q + 1), wrow);
      else if constexpr (kHalf) pipe.fetch<64, 2>(w + 64 * kFull, wrow);
      else next_tap();
      steps(a + 64 * q, std::integral_constant<int, 4>{});
    }
    if constexpr (kHalf) {
      pipe.commit<64, 2>();
      next_tap();
      steps(a + 64 * kFull, std::integral_constant<int, 2>{});
    }
  }
  __syncthreads();
  auto gradient = [&](int layer) __attribute__((always_inline)) {
    each_quad<1, 2>(acc, ln, [&](int, int p, int co, floatx4 v) __attribute__((always_inline)) {
      const int64_t o = (min(s0 + g, num_samples - 1) * kPos + p) * 64 + co;
      const floatx4 pre = *reinterpret_cast<const floatx4*>(net.pre[layer] + o);
      bf16x4n h;
#pragma unroll
      for (int i = 0; i < 4; ++i) h[i] = static_cast<__bf16>(v[i] * gelu_grad(pre[i]));
      if (layer > 0) *reinterpret_cast<bf16x4n*>(act + g * kActElems + act_at(p, co)) = h;
      if (s0 + g < num_samples) *reinterpret_cast<bf16x4n*>(net.dz[layer] + o) = h;
    });
    __syncthreads();
  };
  gradient(2);
  zero_tiles<1, 2>(acc);
  conv_channels<1, 2, 4>(act, pipe, net.wt[1], kTaps * 64, 64, kDil3, ln, acc,
                         [&]() __attribute__((always_inline)) { pipe.fetch<64, 4>(net.wt[0], kTaps * 64); });
  __syncthreads();
  gradient(1);
  zero_tiles<1, 2>(acc);
  conv_channels<1, 2, 4>(act, pipe, net.wt[0], kTaps * 64, 64, kDil2, ln, acc, [] {});
  gradient(0);
}

// Tiles per wavefront of the estimator: one (two samples a workgroup, four workgroups a CU, so eight samples a
// CU at a time) or two (four samples, three workgroups, twelve), whichever takes the shorter rounds: a full round of
// one takes 0.79 of the time of two.  224 output channels, one and two: 2048 samples 77 and 78 us, 2052 109 and 91,
// 3072 121 and 99, 3300 131 and 147, 4096 152 and 158, 5000 195 and 180, 16384 592 and 534.  The training forward pass,
// which stores what the backward pass needs, takes one tile at every size: 2052 samples 128 and 123 us, 3072 159 and 235,
// 4096 214 and 321, 16384 788 and 1199.
int fused_tiles(int64_t samples) {
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess)
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 256;
  const auto rounds = [&](int64_t a_round) { return static_cast<double>((samples + a_round - 1) / a_round); };
  return 0.79 * rounds(8 * cus) <= rounds(12 * cus) ? 1 : 2;
}

unsigned blocks_for(int64_t n) { return static_cast<unsigned>((n + 255) / 256); }

}  // namespace

extern "C" int hpx_conv1d_forward(const uint16_t* in, int64_t num_samples, int cin, int taps, int dilation,
                                  const uint16_t* weight, const float* bias, int cout, int mode, float* out_f32,
                                  uint16_t* out_bf16, void* stream) {
  HPX_REQUIRE(dilation >= 1 && dilation < kPos, "hpx_conv1d_forward: dilation must be in [1, 63]");
  HPX_REQUIRE(num_samples >= 0 && num_samples <= 0x7fffffff, "hpx_conv1d_forward: invalid sample count");
  HPX_REQUIRE(cout >= 32 && cout % 32 == 0, "hpx_conv1d_forward: cout must be a multiple of 32 (got %d)", cout);
  HPX_REQUIRE(mode >= 0 && mode <= 2, "hpx_conv1d_forward: mode must be 0 (linear), 1 (GELU) or 2 (accumulate)");
  if (num_samples == 0) return HPX_OK;
  HPX_REQUIRE(in && weight && (out_f32 || out_bf16) && (mode != 2 || out_f32), "hpx_conv1d_forward: null pointer");
  const dim3 g(static_cast<unsigned>(num_samples));
  const hipStream_t s = as_stream(stream);
#define HPX_CONV(CIN, TAPS) \
  hipLaunchKernelGGL((conv_fwd_kernel<CIN, TAPS>), g, dim3(256), 0, s, in, weight, bias, cout, dilation, mode, \
                     out_f32, out_bf16)
  if (cin == 8 && taps == kTaps) HPX_CONV(8, kTaps);
  else if (cin == 8 && taps == kSkipTaps) HPX_CONV(8, kSkipTaps);
  else if (cin == 64 && taps == kTaps) HPX_CONV(64, kTaps);
  else if (cin == 224 && taps == kTaps) HPX_CONV(224, kTaps);
  else {
    set_error("hpx_conv1d_forward: (cin %d, taps %d) not instantiated ((8|64|224, 5), (8, 17))", cin, taps);
    return HPX_ERR_UNSUPPORTED;
  }
#undef HPX_CONV
  return check_launch("hpx_conv1d_forward");
}

extern "C" int64_t hpx_conv1d_wgrad_workspace(int64_t num_samples, int cin, int cout, int taps) {
  const int64_t chunks = (num_samples + kWgSamples - 1) / kWgSamples;
  return chunks * static_cast<int64_t>(cout) * (static_cast<int64_t>(taps) * cin + 1) *
         static_cast<int64_t>(sizeof(float));
}

extern "C" int hpx_conv1d_wgrad(const uint16_t* dz, const uint16_t* in, int64_t num_samples, int cin, int cout,
                                int taps, int dilation, float* workspace, float* grad_weight, float* grad_bias,
                                void* stream) {
  HPX_REQUIRE(dilation >= 1 && dilation < kPos, "hpx_conv1d_wgrad: dilation must be in [1, 63]");
  HPX_REQUIRE(num_samples >= 1 && num_samples <= 0x7fffffff && cin >= 1 && cout >= 1 && taps >= 1 && (taps & 1) &&
                  taps < kPos,
              "hpx_conv1d_wgrad: invalid sizes");
  HPX_REQUIRE(dz && in && workspace && grad_weight && grad_bias, "hpx_conv1d_wgrad: null pointer");
  const int chunks = static_cast<int>((num_samples + kWgSamples - 1) / kWgSamples);
  const int64_t nw = static_cast<int64_t>(cout) * taps * cin;
  float* part_w = workspace;
  float* part_b = workspace + static_cast<int64_t>(chunks) * nw;
  const hipStream_t s = as_stream(stream);
  const dim3 g(static_cast<unsigned>(chunks), static_cast<unsigned>((cout + 31) / 32),
               static_cast<unsigned>((taps * cin + 63) / 64));
  // Matrix-core form where the operands are whole 16-byte vectors and whole 32-channel tiles; it
  // is the faster one for every such size, the VALU form serves the others, with the same bits.
  const bool aligned = ((reinterpret_cast<uintptr_t>(dz) | reinterpret_cast<uintptr_t>(in)) & 15u) == 0;
  if (aligned && cout % 32 == 0 && cin % 8 == 0 && cin <= 64) {
    const auto launch = [&](auto kernel, int cot) {
      const int tiles = (2 * cot * (taps * cin / 16 + 1) + 3) / 4, waves = wgrad_waves(cot);
      hipLaunchKernelGGL(kernel, dim3(chunks, cout / (32 * cot), (tiles + waves - 1) / waves), dim3(64 * waves),
                         kPos * (wgrad_dz_stride(cot) + 2 * kWgXStride) * sizeof(uint16_t), s, dz, in,
                         static_cast<int>(num_samples), cout, cin, taps, dilation, part_w, part_b);
    };
    if (cout % 224 == 0) launch(wgrad_mfma_kernel<7>, 7);
    else if (cout % 64 == 0) launch(wgrad_mfma_kernel<2>, 2);
    else launch(wgrad_mfma_kernel<1>, 1);
  } else {
    hipLaunchKernelGGL(wgrad_kernel, g, dim3(256), 0, s, dz, in, static_cast<int>(num_samples), cout, cin, taps,
                       dilation, part_w, part_b);
  }
  hipLaunchKernelGGL(reduce_parts_kernel, dim3(blocks_for(nw + cout)), dim3(256), 0, s, part_w,
                     nw, part_b, static_cast<int64_t>(cout), chunks, grad_weight, grad_bias);
  return check_launch("hpx_conv1d_wgrad");
}

extern "C" int hpx_gelu_backward(const float* grad, const float* pre, int64_t n, uint16_t* dz, void* stream) {
  HPX_REQUIRE(n >= 0, "hpx_gelu_backward: negative size");
  if (n == 0) return HPX_OK;
  HPX_REQUIRE(grad && pre && dz, "hpx_gelu_backward: null pointer");
  hipLaunchKernelGGL(gelu_bwd_kernel, dim3(blocks_for(n)), dim3(256), 0, as_stream(stream), grad, pre, n, dz);
  return check_launch("hpx_gelu_backward");
}

extern "C" int hpx_to_bf16(const float* x, int64_t n, uint16_t* y, void* stream) {
  HPX_REQUIRE(n >= 0, "hpx_to_bf16: negative size");
  if (n == 0) return HPX_OK;
  HPX_REQUIRE(x && y, "hpx_to_bf16: null pointer");
  hipLaunchKernelGGL(to_bf16_kernel, dim3(blocks_for(n)), dim3(256), 0, as_stream(stream), x, n, y);
  return check_launch("hpx_to_bf16");
}

extern "C" int hpx_net_input(const hpx_c64* ls, int64_t num_drops, int num_rx, int num_tx, int pilot_words, int cin,
                             const double* noise_power, uint16_t* x, void* stream) {
  HPX_REQUIRE(num_drops >= 0 && num_drops <= 0x7fffffff && num_rx >= 1 && num_tx >= 1 && pilot_words >= 1 &&
                  cin >= 2 * pilot_words + 2,
              "hpx_net_input: invalid sizes");
  const int64_t samples = static_cast<int64_t>(num_tx) * num_drops * num_rx;
  if (samples == 0) return HPX_OK;
  HPX_REQUIRE(ls && x, "hpx_net_input: null pointer");
  hipLaunchKernelGGL(net_input_kernel, dim3(blocks_for(samples * kPos)), dim3(256), 0, as_stream(stream),
                     reinterpret_cast<const float2*>(ls), samples, static_cast<int>(num_drops), num_rx, pilot_words,
                     cin, noise_power, x);
  return check_launch("hpx_net_input");
}

extern "C" int hpx_net_output(const float* out, int64_t num_samples, int words, int num_subcarriers, hpx_c64* est,
                              void* stream) {
  HPX_REQUIRE(num_samples >= 0 && words >= 1 && num_subcarriers >= kPos && num_subcarriers % kPos == 0,
              "hpx_net_output: subcarriers must be a multiple of %d", kPos);
  if (num_samples == 0) return HPX_OK;
  HPX_REQUIRE(out && est, "hpx_net_output: null pointer");
  const int64_t n = num_samples * words * num_subcarriers;
  hipLaunchKernelGGL(net_output_kernel, dim3(blocks_for(n)), dim3(256), 0, as_stream(stream), out, num_samples, words,
                     num_subcarriers, reinterpret_cast<float2*>(est));
  return check_launch("hpx_net_output");
}

extern "C" int hpx_estimate_error(const hpx_c64* est, const hpx_c64* csi, const hpx_c64* spatial, int64_t num_drops,
                                  int num_rx, int num_tx, int64_t grid_elements, double* err, double* power,
                                  void* stream) {
  HPX_REQUIRE(num_drops >= 0 && num_drops <= 0x7fffffff && num_rx >= 1 && num_tx >= 1 && grid_elements >= 1,
              "hpx_estimate_error: invalid sizes");
  const int64_t samples = static_cast<int64_t>(num_tx) * num_drops * num_rx;
  if (samples == 0) return HPX_OK;
  HPX_REQUIRE(est && csi && spatial && err && power, "hpx_estimate_error: null pointer");
  HPX_REQUIRE(samples <= 0x7fffffff, "hpx_estimate_error: too many samples");
  hipLaunchKernelGGL(estimate_error_kernel, dim3(static_cast<unsigned>(samples)), dim3(256), 0, as_stream(stream),
                     reinterpret_cast<const float2*>(est), reinterpret_cast<const float2*>(csi),
                     reinterpret_cast<const float2*>(spatial), static_cast<int>(num_drops), num_rx, num_tx,
                     grid_elements, err, power);
  return check_launch("hpx_estimate_error");
}

namespace {

template <class GRAD>
int nmse_grad(const char* name, const float* out, const hpx_c64* csi, const hpx_c64* spatial, int64_t num_drops, int num_rx,
              int num_tx, int words, int num_subcarriers, const int32_t* group, int num_groups, double* work, GRAD* grad,
              double* loss, void* stream) {
  HPX_REQUIRE(num_drops >= 1 && num_drops <= 0x7fffffff && num_rx >= 1 && num_tx >= 1 && words >= 1 &&
                  num_subcarriers >= kPos && num_subcarriers % kPos == 0 && num_groups >= 1 && (group || num_groups == 1),
              "%s: invalid sizes", name);
  HPX_REQUIRE(out && csi && spatial && work && grad && loss, "%s: null pointer", name);
  const int64_t samples = static_cast<int64_t>(num_tx) * num_drops * num_rx;
  HPX_REQUIRE(samples <= 0x7fffffff, "%s: too many samples", name);
  const hipStream_t s = as_stream(stream);
  const auto* c = reinterpret_cast<const float2*>(csi);
  const auto* sp = reinterpret_cast<const float2*>(spatial);
  const int nd = static_cast<int>(num_drops);
  const dim3 g(static_cast<unsigned>(samples));
  // work[0 .. 2 num_groups) must be zero on entry
  hipLaunchKernelGGL(loss_accumulate_kernel, g, dim3(256), 0, s, out, c, sp, nd, num_rx, num_tx, words, num_subcarriers,
                     group, num_groups, work);
  hipLaunchKernelGGL(loss_finish_kernel, dim3(1), dim3(64), 0, s, num_groups, work, loss);
  // Few samples in shares, up to 1024 workgroups (four a CU): the whole call with one sample of 57344 pairs 103 us in
  // one workgroup, 61 in shares, with 16 of 573440 1679 and 939 us; from 1024 samples on each is one share.  A sample
  // of 64 pairs is one wavefront.
  const int64_t pairs = static_cast<int64_t>(words) * num_subcarriers;
  const int64_t threads = std::min<int64_t>(256, (pairs + 63) / 64 * 64);
  const dim3 gs(g.x, static_cast<unsigned>(std::max<int64_t>(1, std::min((pairs + threads - 1) / threads, 1024 / samples))));
  hipLaunchKernelGGL((loss_grad_kernel<GRAD>), gs, dim3(static_cast<unsigned>(threads)), 0, s, out, c, sp, nd, num_rx, num_tx, words, num_subcarriers,
                     group, num_groups, work, grad);
  return check_launch(name);
}

}  // namespace

extern "C" int hpx_nmse_grad(const float* out, const hpx_c64* csi, const hpx_c64* spatial, int64_t num_drops,
                             int num_rx, int num_tx, int words, int num_subcarriers, const int32_t* group,
                             int num_groups, double* work, float* grad, double* loss, void* stream) {
  return nmse_grad("hpx_nmse_grad", out, csi, spatial, num_drops, num_rx, num_tx, words, num_subcarriers, group,
                   num_groups, work, grad, loss, stream);
}

extern "C" int hpx_nmse_grad_bf16(const float* out, const hpx_c64* csi, const hpx_c64* spatial, int64_t num_drops,
                                  int num_rx, int num_tx, int words, int num_subcarriers, const int32_t* group,
                                  int num_groups, double* work, uint16_t* grad, double* loss, void* stream) {
  return nmse_grad("hpx_nmse_grad_bf16", out, csi, spatial, num_drops, num_rx, num_tx, words, num_subcarriers, group,
                   num_groups, work, grad, loss, stream);
}

extern "C" int hpx_net_forward(const uint16_t* x, int64_t num_samples, const uint16_t* const* weights,
                               const float* const* biases, int cout, float* const* pre, uint16_t* const* act, float* out,
                               void* stream) {
  HPX_REQUIRE(num_samples >= 0 && num_samples <= 0x7fffffff, "hpx_net_forward: invalid sample count");
  HPX_REQUIRE(cout >= 32 && cout % 32 == 0, "hpx_net_forward: cout must be a multiple of 32 (got %d)", cout);
  if (num_samples == 0) return HPX_OK;
  HPX_REQUIRE(x && weights && biases && pre && act && out, "hpx_net_forward: null pointer");
  NetWeights net;
  Kept kept;
  kept.out = out;
  uintptr_t all = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out);
  for (int i = 0; i < 5; ++i) {
    HPX_REQUIRE(weights[i] && biases[i], "hpx_net_forward: null layer %d", i);
    net.w[i] = weights[i];
    net.b[i] = biases[i];
  }
  for (int i = 0; i < 3; ++i) {
    HPX_REQUIRE(pre[i] && act[i], "hpx_net_forward: null layer %d", i);
    kept.pre[i] = pre[i];
    kept.act[i] = act[i];
    all |= reinterpret_cast<uintptr_t>(pre[i]) | reinterpret_cast<uintptr_t>(act[i]);
  }
  HPX_REQUIRE((all & 15u) == 0, "hpx_net_forward: arrays must be 16-byte aligned");
  hipLaunchKernelGGL((net_forward_kernel<1, true, true>), dim3(static_cast<unsigned>((num_samples + 1) / 2)), dim3(256), 0,
                     as_stream(stream), static_cast<const float2*>(nullptr), 0, 0, 0, 0, static_cast<const int32_t*>(nullptr),
                     static_cast<const float2*>(nullptr), 0, static_cast<const double*>(nullptr), x, num_samples, net, cout,
                     static_cast<float*>(nullptr), kept);
  return check_launch("hpx_net_forward");
}

extern "C" int hpx_net_backward(const uint16_t* dz_out, int64_t num_samples, int cout, const uint16_t* const* weights_transposed,
                                const float* const* pre, uint16_t* const* dz, void* stream) {
  HPX_REQUIRE(num_samples >= 0 && num_samples <= 0x7fffffff, "hpx_net_backward: invalid sample count");
  if (cout != 64 && cout != 224) {  // (as the layer-by-layer backward convolution)
    set_error("hpx_net_backward: cout %d not instantiated (64, 224)", cout);
    return HPX_ERR_UNSUPPORTED;
  }
  if (num_samples == 0) return HPX_OK;
  HPX_REQUIRE(dz_out && weights_transposed && pre && dz, "hpx_net_backward: null pointer");
  Gradients net;
  uintptr_t all = reinterpret_cast<uintptr_t>(dz_out);
  for (int i = 0; i < 3; ++i) {
    HPX_REQUIRE(weights_transposed[i] && pre[i] && dz[i], "hpx_net_backward: null layer %d", i);
    net.wt[i] = weights_transposed[i];
    net.pre[i] = pre[i];
    net.dz[i] = dz[i];
    all |= reinterpret_cast<uintptr_t>(net.wt[i]) | reinterpret_cast<uintptr_t>(pre[i]) | reinterpret_cast<uintptr_t>(dz[i]);
  }
  HPX_REQUIRE((all & 15u) == 0, "hpx_net_backward: arrays must be 16-byte aligned");
  hipLaunchKernelGGL(cout == 64 ? net_backward_kernel<64> : net_backward_kernel<224>, dim3(static_cast<unsigned>((num_samples + 1) / 2)), dim3(256), 0,
                     as_stream(stream), dz_out, num_samples, net);
  return check_launch("hpx_net_backward");
}

extern "C" int hpx_adam_steps(const hpx_adam_tensor* tensors, int count, float lr, float beta1, float beta2, float eps,
                              int64_t step, void* stream) {
  HPX_REQUIRE(count >= 0 && count <= HPX_ADAM_MAX_TENSORS && step >= 1, "hpx_adam_steps: invalid arguments");
  AdamTensors a{};
  int64_t blocks = 0;
  for (int i = 0; i < count; ++i) {
    const hpx_adam_tensor& t = tensors[i];
    HPX_REQUIRE(t.n >= 0 && (t.n == 0 || (t.param && t.grad && t.m1 && t.m2)), "hpx_adam_steps: invalid tensor %d", i);
    HPX_REQUIRE(!t.weight_transposed || (t.cin >= 1 && t.taps >= 1 && t.n % (static_cast<int64_t>(t.cin) * t.taps) == 0),
                "hpx_adam_steps: tensor %d is not [cout][taps][cin]", i);
    a.t[i] = t;
    a.first_block[i] = static_cast<int>(blocks);
    blocks += (t.n + 255) / 256;
    HPX_REQUIRE(blocks <= 0x7fffffff, "hpx_adam_steps: too many parameters");
  }
  a.count = count;
  a.first_block[count] = static_cast<int>(blocks);
  if (blocks == 0) return HPX_OK;
  const float c1 = static_cast<float>(1.0 - pow(static_cast<double>(beta1), static_cast<double>(step)));
  const float c2 = static_cast<float>(1.0 - pow(static_cast<double>(beta2), static_cast<double>(step)));
  hipLaunchKernelGGL(adam_tensors_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, as_stream(stream), a, lr, beta1,
                     beta2, eps, c1, c2);
  return check_launch("hpx_adam_steps");
}

extern "C" int hpx_adam_step(float* param, const float* grad, float* m1, float* m2, int64_t n, float lr, float beta1,
                             float beta2, float eps, int64_t step, void* stream) {
  HPX_REQUIRE(n >= 0 && step >= 1, "hpx_adam_step: invalid arguments");
  if (n == 0) return HPX_OK;
  HPX_REQUIRE(param && grad && m1 && m2, "hpx_adam_step: null pointer");
  const float c1 = static_cast<float>(1.0 - pow(static_cast<double>(beta1), static_cast<double>(step)));
  const float c2 = static_cast<float>(1.0 - pow(static_cast<double>(beta2), static_cast<double>(step)));
  hipLaunchKernelGGL(adam_kernel, dim3(blocks_for(n)), dim3(256), 0, as_stream(stream), param, grad, m1, m2, n, lr,
                     beta1, beta2, eps, c1, c2);
  return check_launch("hpx_adam_step");
}

extern "C" int hpx_conv1d_weight_copies(const float* param, int cout, int cin, int taps, uint16_t* weight,
                                        uint16_t* weight_transposed, void* stream) {
  HPX_REQUIRE(cout >= 1 && cin >= 1 && taps >= 1, "hpx_conv1d_weight_copies: invalid sizes");
  HPX_REQUIRE(param && (weight || weight_transposed), "hpx_conv1d_weight_copies: null pointer");
  const int64_t n = static_cast<int64_t>(cout) * taps * cin;
  hipLaunchKernelGGL(weight_copies_kernel, dim3(blocks_for(n)), dim3(256), 0, as_stream(stream), param, cout, cin,
                     taps, weight, weight_transposed);
  return check_launch("hpx_conv1d_weight_copies");
}

extern "C" int hpx_learned_estimate(const hpx_c64* grid, int64_t num_drops, int num_rx, int num_tx, int words,
                                    int num_subcarriers, const int32_t* pilot_index, const hpx_c64* pilot_values,
                                    int num_pilots, const double* noise_power, const uint16_t* const* weights,
                                    const float* const* biases, int cout, hpx_c64* est, void* stream) {
  HPX_REQUIRE(num_drops >= 0 && num_drops <= 0x7fffffff && num_rx >= 1 && num_tx >= 1 && words >= 1,
              "hpx_learned_estimate: invalid sizes");
  HPX_REQUIRE(num_subcarriers >= kPos && num_subcarriers % kPos == 0 && num_pilots >= kPos && num_pilots % kPos == 0 &&
                  2 * (num_pilots / kPos) + 2 <= 8,
              "hpx_learned_estimate: needs 64-position pilot words (at most 3) and a multiple of 64 subcarriers");
  HPX_REQUIRE(cout == 2 * words * (num_subcarriers / kPos) && cout % 32 == 0,
              "hpx_learned_estimate: output channels %d do not match the grid", cout);
  const int64_t samples = static_cast<int64_t>(num_tx) * num_drops * num_rx;
  if (samples == 0) return HPX_OK;
  HPX_REQUIRE(grid && pilot_index && pilot_values && weights && biases && est, "hpx_learned_estimate: null pointer");
  for (int i = 0; i < 5; ++i) HPX_REQUIRE(weights[i] && biases[i], "hpx_learned_estimate: null layer %d", i);
  const int pt = fused_tiles(samples);
  const int64_t blocks = (samples + 2 * pt - 1) / (2 * pt);
  HPX_REQUIRE(blocks <= 0x7fffffff, "hpx_learned_estimate: too many samples");
  NetWeights net;
  for (int i = 0; i < 5; ++i) {
    net.w[i] = weights[i];
    net.b[i] = biases[i];
  }
  const bool vec = (num_subcarriers / kPos) % 2 == 0 && (reinterpret_cast<uintptr_t>(est) & 15u) == 0;
#define HPX_ESTIMATE(PT, VEC)                                                                                          \
  hipLaunchKernelGGL((net_forward_kernel<PT, false, VEC>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0,          \
                     as_stream(stream), reinterpret_cast<const float2*>(grid), static_cast<int>(num_drops), num_rx,    \
                     words, num_subcarriers, pilot_index, reinterpret_cast<const float2*>(pilot_values), num_pilots,   \
                     noise_power, static_cast<const uint16_t*>(nullptr), samples, net, cout,                           \
                     reinterpret_cast<float*>(est), Kept{})
  if (vec) {
    if (pt == 2) HPX_ESTIMATE(2, true);
    else HPX_ESTIMATE(1, true);
  } else {
    if (pt == 2) HPX_ESTIMATE(2, false);
    else HPX_ESTIMATE(1, false);
  }
#undef HPX_ESTIMATE
  return check_launch("hpx_learned_estimate");
}
