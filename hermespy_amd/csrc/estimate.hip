// Pilot-based channel estimation and detection on estimated channels.
//
//   hpx_pilot_ls          least squares at every stream's pilots
//                         (hermespy/modem/waveforms/orthogonal/channel.py:44-48)
//   hpx_lmmse_apply       linear MMSE interpolation of the pilot LS values over the
//                         whole grid with a precomputed filter (a complex float32 GEMM)
//   hpx_detect_estimated  ZF/MMSE detection of the data elements from estimated channels,
//                         hard demapping and per-drop bit errors against the Philox bits
//                         (waveform.py:235-250, psk_qam_mapping.py:171-259, evaluators.py:239-258)
#include <math.h>

#include <algorithm>

#include "hpx_common.hpp"
#include "hpx_detect.hpp"
#include "hpx_mapping.hpp"

using namespace hpx;

namespace {

constexpr int kMaxRx = 8;

inline hipStream_t as_stream(void* s) { return static_cast<hipStream_t>(s); }

__global__ void __launch_bounds__(256) pilot_ls_kernel(const float2* __restrict__ grid, int64_t total, int num_drops,
                                                       int num_rx, int64_t grid_elements, int num_pilots,
                                                       const int32_t* __restrict__ pidx,
                                                       const float2* __restrict__ pval, float2* __restrict__ ls) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= total) return;
  // ls[t][d][r][j]
  const int j = static_cast<int>(i % num_pilots);
  const int64_t rest = i / num_pilots;
  const int64_t dr = rest % (static_cast<int64_t>(num_drops) * num_rx);
  const int t = static_cast<int>(rest / (static_cast<int64_t>(num_drops) * num_rx));
  const float2 x = pval[t * num_pilots + j];
  const float2 y = grid[dr * grid_elements + pidx[t * num_pilots + j]];
  ls[i] = cscale(cmulc(x, y), 1.0f / cabs2(x));  // y / x
}

// est[t][row][e] = sum_j W[t][e][j] ls[t][row][j] for the rows of several filter sets (SNR points), each
// with its own filter.  One complex product is four real ones on float32 MFMA (32x32x2): rows of ls
// are the A operand, grid elements the B operand, so a wavefront's lanes hold consecutive elements
// of a row and store 256 contiguous bytes.  Tile: 64 rows x 128 elements per workgroup (64 x 32 per
// wavefront, real and imaginary accumulators), K chunks of 32 staged in LDS with the next chunk's
// loads in flight; a lane's 16-byte LDS read holds two pilots, which feed 16 MFMAs per three reads.
// All sets go in one launch (a set alone is a few hundred workgroups), with the row tiles of one
// filter tile next to each other on one XCD, whose L2 then serves the filter.  Bound: float32 MFMA.
// 1000 drops of the 2x2 512-subcarrier link at 11 SNR points (29.4 GFLOP, 0.39 GB): 278 us,
// 106 TFLOP/s (a 32 x 128 FP32 VALU tile and a launch per SNR point took 741 us).  Small calls are latency: the
// contraction's padding and an empty upper half of the rows are left out (one row of 128 pilots and 7168 elements,
// 2 streams: 21.9 us with them, 14.8 without; 100 rows of 16 pilots and 64 elements 12.3 and 7.3, with the VALU tile 9.5).
constexpr int kGemmRows = 64, kGemmCols = 128, kGemmK = 32;
constexpr int kGemmStride = kGemmK + 2;  // float2; rows 16 bytes apart modulo the LDS banks
constexpr int kGemmSets = 16;            // filter sets per launch
constexpr int kXcds = 8;                 // consecutive workgroups go round robin over the XCDs
constexpr int kGemmTiles = (1 << 24) - kXcds;  // tiles per launch: fewer than 2^32 threads
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

struct LmmseSets {
  const int32_t* rows[kGemmSets];
  const float2* filt[kGemmSets];
  int count[kGemmSets];
  int first_tile[kGemmSets + 1];
  int num_sets;
  int begin, end;  // this launch's tiles
};

// VEC: the rows of ls and of the filters are whole 16-byte vectors.
template <bool VEC>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
lmmse_kernel(LmmseSets sets, const float2* __restrict__ ls, int64_t ls_tx_stride,
                                                    int num_pilots, int64_t filt_tx_stride, int64_t elements,
                                                    int col_tiles, float2* __restrict__ est, int64_t est_tx_stride) {
  __shared__ __align__(16) float2 as[kGemmRows * kGemmStride];
  __shared__ __align__(16) float2 bs[kGemmCols * kGemmStride];
  __shared__ int32_t row_of[kGemmRows];  // for the stores (read before the first barrier, not after the last)
  const int per_xcd = (sets.end - sets.begin + kXcds - 1) / kXcds;
  const int tile = sets.begin + static_cast<int>(blockIdx.x % kXcds) * per_xcd + static_cast<int>(blockIdx.x / kXcds);
  if (tile >= sets.end) return;
  int si = 0;
  while (tile >= sets.first_tile[si + 1]) ++si;
  const int count = sets.count[si];
  const int row_tiles = (count + kGemmRows - 1) / kGemmRows;
  int rest = tile - sets.first_tile[si];
  const int r0 = rest % row_tiles * kGemmRows;
  rest /= row_tiles;
  const int64_t e0 = static_cast<int64_t>(rest % col_tiles) * kGemmCols;
  const int t = rest / col_tiles;
  const int32_t* rows = sets.rows[si];
  const float2* lst = ls + t * ls_tx_stride;
  const float2* ft = sets.filt[si] + t * filt_tx_stride;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  // a thread stages pilots 2 (tid % 16), + 1 of rows tid / 16 + 16 i of either operand
  constexpr int kA = kGemmRows / 16, kB = kGemmCols / 16;
  const int kp = 2 * (tid & 15), sr = tid >> 4;
  const float2* arow[kA];
  const float2* brow[kB];
#pragma unroll
  for (int i = 0; i < kA; ++i) {
    const int row = r0 + sr + 16 * i;
    arow[i] = lst + static_cast<int64_t>(rows[row < count ? row : count - 1]) * num_pilots;
  }
#pragma unroll
  for (int i = 0; i < kB; ++i) {
    const int64_t e = e0 + sr + 16 * i;
    brow[i] = ft + (e < elements ? e : elements - 1) * num_pilots;
  }
  if (tid < kGemmRows && r0 + tid < count) row_of[tid] = rows[r0 + tid];
  const bool upper = r0 + 32 < count;  // rows in the upper half of the tile
  floatx4 ra[kA], rb[kB];
  auto pair_at = [&](const float2* row, int k) __attribute__((always_inline)) {
    floatx4 v = {0.f, 0.f, 0.f, 0.f};
    if constexpr (VEC) {
      if (k < num_pilots) v = *reinterpret_cast<const floatx4*>(row + k);
    } else {
      if (k < num_pilots) {
        v[0] = row[k].x;
        v[1] = row[k].y;
      }
      if (k + 1 < num_pilots) {
        v[2] = row[k + 1].x;
        v[3] = row[k + 1].y;
      }
    }
    return v;
  };
  auto load = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kA; ++i) ra[i] = pair_at(arow[i], k0 + kp);
#pragma unroll
    for (int i = 0; i < kB; ++i) rb[i] = pair_at(brow[i], k0 + kp);
  };
  floatx16 re[2], im[2];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int r = 0; r < 16; ++r) re[m][r] = im[m][r] = 0.0f;
  const int mrow = lane & 31, kq = lane >> 5;
  load(0);
  for (int k0 = 0; k0 < num_pilots; k0 += kGemmK) {
#pragma unroll
    for (int i = 0; i < kA; ++i) *reinterpret_cast<floatx4*>(as + (sr + 16 * i) * kGemmStride + kp) = ra[i];
#pragma unroll
    for (int i = 0; i < kB; ++i) *reinterpret_cast<floatx4*>(bs + (sr + 16 * i) * kGemmStride + kp) = rb[i];
    __syncthreads();
    if (k0 + kGemmK < num_pilots) load(k0 + kGemmK);
#pragma unroll
    for (int s = 0; s < kGemmK / 4; ++s) {
      if (k0 + 4 * s >= num_pilots) break;  // (padding)
      const floatx4 b = *reinterpret_cast<const floatx4*>(bs + (32 * wave + mrow) * kGemmStride + 4 * s + 2 * kq);
      floatx4 a[2];
#pragma unroll
      for (int m = 0; m < 2; ++m)
        a[m] = *reinterpret_cast<const floatx4*>(as + (32 * m + mrow) * kGemmStride + 4 * s + 2 * kq);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        if (m && !upper) break;
#pragma unroll
        for (int o = 0; o < 4; o += 2) {
          re[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[m][o], b[o], re[m], 0, 0, 0);
          im[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[m][o], b[o + 1], im[m], 0, 0, 0);
          re[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(-a[m][o + 1], b[o + 1], re[m], 0, 0, 0);
          im[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[m][o + 1], b[o], im[m], 0, 0, 0);
        }
      }
    }
    __syncthreads();
  }
  float2* et = est + t * est_tx_stride;
  const int64_t e = e0 + 32 * wave + mrow;
  if (e >= elements) return;
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = 32 * m + 8 * (r >> 2) + 4 * kq + (r & 3);
      if (r0 + row < count) et[static_cast<int64_t>(row_of[row]) * elements + e] = make_float2(re[m][r], im[m][r]);
    }
}

// bps bits of a stream starting at bit `pos` (LSB-first 32-bit words, four per Philox call)
__device__ __forceinline__ uint32_t stream_symbol_bits(uint64_t seed, uint32_t drop, uint32_t stream, int64_t pos,
                                                       int bps) {
  const int64_t wi = pos >> 5;
  const uint4 r = stream_call(seed, drop, stream, static_cast<uint32_t>(wi >> 2));
  const uint32_t comp[4] = {r.x, r.y, r.z, r.w};
  uint64_t v = comp[wi & 3];
  const int sh = static_cast<int>(pos & 31);
  if (sh + bps > 32) {
    const int64_t wn = wi + 1;
    uint32_t next;
    if ((wn & 3) != 0) {
      next = comp[wn & 3];
    } else {
      const uint4 q = stream_call(seed, drop, stream, static_cast<uint32_t>(wn >> 2));
      next = q.x;
    }
    v |= static_cast<uint64_t>(next) << 32;
  }
  return static_cast<uint32_t>(v >> sh) & ((1u << bps) - 1u);
}

// Workgroup: drop d, a share of its words.  The transmitted bits of these words are drawn once into LDS
// (bits_words words per stream, 0 where they would not fit; an element that lies outside them draws its
// own, which cost a Philox call per element and stream), decisions compare float32 values with the
// float32 boundaries (the decisions of the float64 demapper), and an element's word and subcarrier are
// carried along instead of divided out.  Shares of a drop add their errors to errors[d], zero before.
// 1000 drops of the 2x2 512-subcarrier link, 16-QAM: 127 us (3.6 TB/s) before, 102 us (4.5 TB/s) now.
template <int NT, int PAM>
__global__ void __launch_bounds__(256) detect_estimated_kernel(
    const float2* __restrict__ grid, const float2* __restrict__ est, int num_drops, int num_rx, int words, int n,
    const int32_t* __restrict__ elements, const int32_t* __restrict__ word_data, int bps, DemapBounds bounds, int mmse,
    const double* __restrict__ noise_power, uint64_t seed, int64_t first_drop, int data_total, int segs, int bits_words,
    int32_t* __restrict__ errors, float2* __restrict__ equalized) {
  extern __shared__ __align__(16) uint32_t bits[];  // [NT][bits_words]
  __shared__ int red[4];
  const int d = static_cast<int>(blockIdx.x) / segs, seg = static_cast<int>(blockIdx.x) - d * segs;
  const uint32_t drop = static_cast<uint32_t>(first_drop + d);
  const int64_t wn = static_cast<int64_t>(words) * n;
  const int w_begin = static_cast<int>(static_cast<int64_t>(words) * seg / segs);
  const int w_end = static_cast<int>(static_cast<int64_t>(words) * (seg + 1) / segs);
  const float s2 = mmse ? static_cast<float>(noise_power[d]) : 0.0f;
  const float2* yd = grid + static_cast<int64_t>(d) * num_rx * wn;
  auto data_before = [&](int w) { return !word_data ? static_cast<int64_t>(w) * n : w < words ? word_data[w] : data_total; };
  // the share's bits: whole Philox calls from the one that holds its first bit
  const int64_t call0 = (data_before(w_begin) * bps) >> 7;
  const int64_t end = data_before(w_end) * bps;
  const int calls = static_cast<int>(std::max<int64_t>(0, std::min<int64_t>(((end + 127) >> 7) - call0, bits_words / 4)));
  for (int i = threadIdx.x; i < NT * calls; i += 256) {
    const int t = i / calls, c = i - t * calls;
    *reinterpret_cast<uint4*>(bits + t * bits_words + 4 * c) =
        stream_call(seed, drop, HPX_STREAM_BITS + t, static_cast<uint32_t>(call0 + c));
  }
  __syncthreads();
  float ta[PAM / 2], tb[PAM / 2];
#pragma unroll
  for (int i = 0; i < PAM / 2; ++i) {
    ta[i] = bounds.a[i];
    tb[i] = bounds.b[i];
  }
  int err = 0;
  const int dw = 256 / n, dq = 256 - dw * n;
  int w = w_begin + static_cast<int>(threadIdx.x) / n, q = static_cast<int>(threadIdx.x) % n;
  for (; w < w_end; w += dw, q += dq) {
    if (q >= n) {
      q -= n;
      if (++w >= w_end) break;
    }
    const int64_t e = static_cast<int64_t>(w) * n + q;
    const int el = elements ? elements[e] : q;
    if (el < 0) continue;
    const int gidx = (word_data ? word_data[w] : w * n) + el;
    float2 x[NT];
    detect_rows<NT>(
        num_rx,
        [&](int r, int t) { return est[((static_cast<int64_t>(t) * num_drops + d) * num_rx + r) * wn + e]; },
        [&](int r) { return yd[r * wn + e]; }, s2, x);
    const int64_t pos = static_cast<int64_t>(gidx) * bps;
    const int64_t at = pos - 128 * call0;
    const bool drawn = at >= 0 && at + bps <= 128 * static_cast<int64_t>(calls);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const uint32_t rx = demap_symbol_f32_reg<PAM>(x[t].x, x[t].y, ta, tb);
      uint32_t tx;
      if (drawn) {
        const uint32_t* bw = bits + t * bits_words + static_cast<int>(at >> 5);
        const int sh = static_cast<int>(at) & 31;
        uint64_t v = bw[0];
        if (sh + bps > 32) v |= static_cast<uint64_t>(bw[1]) << 32;
        tx = static_cast<uint32_t>(v >> sh) & ((1u << bps) - 1u);
      } else {
        tx = stream_symbol_bits(seed, drop, HPX_STREAM_BITS + t, pos, bps);
      }
      err += __popc(rx ^ tx);
      if (equalized) equalized[(static_cast<int64_t>(d) * NT + t) * data_total + gidx] = x[t];
    }
  }
  for (int off = 32; off > 0; off >>= 1) err += __shfl_down(err, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = err;
  __syncthreads();
  if (threadIdx.x == 0) {
    err = (red[0] + red[1]) + (red[2] + red[3]);
    if (segs == 1) errors[d] = err;
    else if (err) atomicAdd(errors + d, err);
  }
}

__global__ void __launch_bounds__(256) zero_counts_kernel(int32_t* __restrict__ errors, int count) {
  const int i = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
  if (i < count) errors[i] = 0;
}

// Shares of a drop.  A launch whose arrays stay in the 256 MB memory-side cache to a good part is bounded by
// latency and takes shares up to 4096 workgroups; one that streams from HBM only two workgroups a CU, at least
// one a drop: a 2x2 512-subcarrier link with one and with more shares, 11 drops 63 and 15 us, 400 (183 MB)
// 55 and 34, 600 (275 MB) 73 and 51, 1000 (459 MB) 102 and 109.  The line lies between the last two.
// A share has at least a workgroup's threads of elements, and drops of a few steps are not cut: 200 drops of 14
// words of 64 subcarriers, one stream 7.7 us with a workgroup a drop, 12.5 in 14 shares each, 5.3 whole; two streams 11.7,
// 13.9 and in four shares 8.8; eight streams 59, 72 and 35.
int detect_segments(int64_t drops, int64_t drop_bytes, int words, int64_t elements, int streams) {
  if (elements * streams <= 1024) return 1;
  const int64_t target = drops * drop_bytes <= (int64_t(384) << 20) ? 4096 : 512;
  const int64_t most = std::min<int64_t>(words, (elements + 255) / 256);
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(most, target / std::max<int64_t>(drops, 1))));
}

template <int NT>
int detect_launch(const Modulation& mod, const float2* grid, const float2* est, int num_drops, int num_rx, int words, int n,
                  const int32_t* elements, const int32_t* word_data, int mmse, const double* noise_power, uint64_t seed,
                  int64_t first_drop, int data_total, int32_t* errors, float2* equalized, hipStream_t stream) {
  const int64_t per_drop = static_cast<int64_t>(words) * n;
  const int segs = detect_segments(num_drops, 8 * per_drop * (num_rx + num_rx * NT + NT), words, per_drop, NT);
  // (a share holds at most this many bits a stream, and begins inside a call)
  const int64_t share = static_cast<int64_t>((words + segs - 1) / segs) * n * mod.bps;
  const int64_t want = 4 * ((share + 127) / 128 + 1);
  const int bits_words = want * NT * 4 <= 48 * 1024 ? static_cast<int>(want) : 0;
  const DemapBounds& bounds = demap_bounds_of(mod);
  if (segs > 1)
    hipLaunchKernelGGL(zero_counts_kernel, dim3(static_cast<unsigned>((num_drops + 255) / 256)), dim3(256), 0, stream, errors,
                       num_drops);
#define HPX_DETECT_PAM(PAM)                                                                                                \
  hipLaunchKernelGGL((detect_estimated_kernel<NT, PAM>), dim3(static_cast<unsigned>(static_cast<int64_t>(num_drops) * segs)), dim3(256),          \
                     static_cast<size_t>(bits_words) * NT * 4, stream, grid, est, num_drops, num_rx, words, n, elements,   \
                     word_data, mod.bps, bounds, mmse, noise_power, seed, first_drop, data_total, segs, bits_words,        \
                     errors, equalized)
  switch (mod.pam) {
    case 2: HPX_DETECT_PAM(2); break;
    case 4: HPX_DETECT_PAM(4); break;
    case 8: HPX_DETECT_PAM(8); break;
    default: HPX_DETECT_PAM(16); break;
  }
#undef HPX_DETECT_PAM
  return check_launch("hpx_detect_estimated");
}

// The sets' tiles in launches of up to kGemmSets sets; filter of set i at filters + i set_stride.
int lmmse_launch(const char* what, const hpx_c64* ls, int num_tx, int64_t num_rows, int num_pilots, const hpx_c64* filters,
                 int64_t set_stride, int64_t elements, const void* const* rows, const int* counts, int num_sets,
                 hpx_c64* est, void* stream) {
  const int64_t col_tiles = (elements + kGemmCols - 1) / kGemmCols;
  HPX_REQUIRE(col_tiles <= 65535, "%s: grid too large", what);
  const bool vec = num_pilots % 2 == 0 &&
                   ((reinterpret_cast<uintptr_t>(ls) | reinterpret_cast<uintptr_t>(filters)) & 15u) == 0;
  auto flush = [&](LmmseSets& sets) -> int {
    if (sets.num_sets == 0) return HPX_OK;
    const int total = sets.first_tile[sets.num_sets];
    for (sets.begin = 0; sets.begin < total; sets.begin = sets.end) {
      sets.end = std::min(total, sets.begin + kGemmTiles);
      const unsigned blocks = static_cast<unsigned>((sets.end - sets.begin + kXcds - 1) / kXcds * kXcds);
      hipLaunchKernelGGL(vec ? lmmse_kernel<true> : lmmse_kernel<false>, dim3(blocks), dim3(256), 0, as_stream(stream), sets,
                         reinterpret_cast<const float2*>(ls), num_rows * num_pilots, num_pilots, elements * num_pilots,
                         elements, static_cast<int>(col_tiles), reinterpret_cast<float2*>(est), num_rows * elements);
    }
    sets.num_sets = 0;
    return check_launch(what);
  };
  LmmseSets sets{};
  for (int i = 0; i < num_sets; ++i) {
    if (counts[i] == 0) continue;
    const int64_t tiles = (static_cast<int64_t>(counts[i]) + kGemmRows - 1) / kGemmRows * col_tiles * num_tx;
    HPX_REQUIRE(tiles <= 0x3fffffff, "%s: grid too large", what);
    if (sets.num_sets == kGemmSets || sets.first_tile[sets.num_sets] + tiles > 0x3fffffff) {
      const int st = flush(sets);
      if (st != HPX_OK) return st;
    }
    const int k = sets.num_sets++;
    sets.rows[k] = static_cast<const int32_t*>(rows[i]);
    sets.filt[k] = reinterpret_cast<const float2*>(filters) + i * set_stride;
    sets.count[k] = counts[i];
    sets.first_tile[0] = 0;
    sets.first_tile[k + 1] = sets.first_tile[k] + static_cast<int>(tiles);
  }
  return flush(sets);
}

}  // namespace

extern "C" int hpx_pilot_ls(const hpx_c64* grid, int64_t num_drops, int num_rx, int num_tx, int64_t grid_elements,
                            int num_pilots, const int32_t* pilot_index, const hpx_c64* pilot_values, hpx_c64* ls,
                            void* stream) {
  HPX_REQUIRE(num_drops >= 0 && num_rx >= 1 && num_tx >= 1 && grid_elements >= 1 && num_pilots >= 1,
              "hpx_pilot_ls: invalid sizes");
  const int64_t total = static_cast<int64_t>(num_tx) * num_drops * num_rx * num_pilots;
  if (total == 0) return HPX_OK;
  HPX_REQUIRE(grid && pilot_index && pilot_values && ls, "hpx_pilot_ls: null pointer");
  HPX_REQUIRE(num_drops <= 0x7fffffff, "hpx_pilot_ls: too many drops");
  hipLaunchKernelGGL(pilot_ls_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0,
                     as_stream(stream), reinterpret_cast<const float2*>(grid), total, static_cast<int>(num_drops),
                     num_rx, grid_elements, num_pilots, pilot_index, reinterpret_cast<const float2*>(pilot_values),
                     reinterpret_cast<float2*>(ls));
  return check_launch("hpx_pilot_ls");
}

extern "C" int hpx_lmmse_apply(const hpx_c64* ls, int num_tx, int64_t num_rows, int num_pilots,
                               const hpx_c64* filter, int64_t elements, const int32_t* rows, int count, hpx_c64* est,
                               void* stream) {
  HPX_REQUIRE(num_tx >= 1 && num_tx <= 65535 && num_rows >= 0 && num_pilots >= 1 && elements >= 1 && count >= 0,
              "hpx_lmmse_apply: invalid sizes");
  if (count == 0) return HPX_OK;
  HPX_REQUIRE(ls && filter && rows && est, "hpx_lmmse_apply: null pointer");
  HPX_REQUIRE(count <= num_rows, "hpx_lmmse_apply: more rows than the LS array holds");
  const void* row_lists[1] = {rows};
  return lmmse_launch("hpx_lmmse_apply", ls, num_tx, num_rows, num_pilots, filter, 0, elements, row_lists, &count, 1, est,
                      stream);
}

extern "C" int hpx_lmmse_apply_sets(const hpx_c64* ls, int num_tx, int64_t num_rows, int num_pilots,
                                    const hpx_c64* filters, int64_t elements, int num_sets,
                                    const int32_t* const* rows_host, const int32_t* counts_host, hpx_c64* est,
                                    void* stream) {
  HPX_REQUIRE(num_tx >= 1 && num_tx <= 65535 && num_rows >= 0 && num_pilots >= 1 && elements >= 1 && num_sets >= 0,
              "hpx_lmmse_apply_sets: invalid sizes");
  if (num_sets == 0) return HPX_OK;
  HPX_REQUIRE(ls && filters && rows_host && counts_host && est, "hpx_lmmse_apply_sets: null pointer");
  for (int i = 0; i < num_sets; ++i) {
    HPX_REQUIRE(counts_host[i] >= 0 && (counts_host[i] == 0 || rows_host[i]), "hpx_lmmse_apply_sets: invalid set %d", i);
    HPX_REQUIRE(counts_host[i] <= num_rows, "hpx_lmmse_apply_sets: more rows than the LS array holds");
  }
  return lmmse_launch("hpx_lmmse_apply_sets", ls, num_tx, num_rows, num_pilots, filters, num_tx * elements * num_pilots,
                      elements, reinterpret_cast<const void* const*>(rows_host), counts_host, num_sets, est, stream);
}

extern "C" int hpx_detect_estimated(const hpx_c64* grid, const hpx_c64* est, int64_t num_drops, int num_rx,
                                    int num_tx, int words, int num_subcarriers, const int32_t* elements,
                                    const int32_t* word_data, int num_data, int modulation_order, int detector,
                                    const double* noise_power, uint64_t seed, int64_t first_drop, int32_t* errors,
                                    hpx_c64* equalized, void* stream) {
  HPX_REQUIRE(num_drops >= 0 && num_drops <= 0x7fffffff && words >= 1 && num_subcarriers >= 1 && num_data >= 0,
              "hpx_detect_estimated: invalid sizes");
  HPX_REQUIRE(detector == HPX_DETECT_ZF || detector == HPX_DETECT_MMSE, "hpx_detect_estimated: unknown detector");
  HPX_REQUIRE(num_rx >= num_tx && num_rx <= kMaxRx, "hpx_detect_estimated: needs num_tx <= num_rx <= %d", kMaxRx);
  HPX_REQUIRE((elements == nullptr) == (word_data == nullptr), "hpx_detect_estimated: give elements and word_data");
  HPX_REQUIRE(elements || num_data == words * num_subcarriers, "hpx_detect_estimated: all-data frame size mismatch");
  HPX_REQUIRE(first_drop >= 0 && first_drop + num_drops <= (int64_t(1) << 32),
              "hpx_detect_estimated: drop index exceeds 32 bits");
  Modulation mod;
  if (modulation_order == 2 || !modulation(modulation_order, 1, &mod)) {
    set_error("hpx_detect_estimated: modulation order %d not supported (4, 16, 64, 256)", modulation_order);
    return HPX_ERR_UNSUPPORTED;
  }
  if (num_drops == 0) return HPX_OK;
  HPX_REQUIRE(grid && est && noise_power && errors, "hpx_detect_estimated: null pointer");
  const hipStream_t s = as_stream(stream);
  const float2* gy = reinterpret_cast<const float2*>(grid);
  const float2* ge = reinterpret_cast<const float2*>(est);
  float2* eq = reinterpret_cast<float2*>(equalized);
  const int nd = static_cast<int>(num_drops);
  const int mm = detector == HPX_DETECT_MMSE;
#define HPX_DETECT_EST(NT)                                                                                        \
  return detect_launch<NT>(mod, gy, ge, nd, num_rx, words, num_subcarriers, elements, word_data, mm, noise_power, \
                           seed, first_drop, num_data, errors, eq, s)
  switch (num_tx) {
    case 1: HPX_DETECT_EST(1);
    case 2: HPX_DETECT_EST(2);
    case 4: HPX_DETECT_EST(4);
    case 8: HPX_DETECT_EST(8);
  }
#undef HPX_DETECT_EST
  set_error("hpx_detect_estimated: num_tx %d not instantiated (1, 2, 4, 8)", num_tx);
  return HPX_ERR_UNSUPPORTED;
}
