// Fused Monte Carlo link drops: one workgroup simulates one drop end to end.
//
// Per drop (prologue):
//   Philox normals -> Phi -> spatial response S = R_rx exp(2 pi j U) R_tx and
//   the SoS table (fading.py:468-499, consistent.py:410-485), Taylor
//   coefficients of every path over the frame, per-word tap means (ideal CSI),
//   twiddles and the constellation table.
// Per OFDM word w (main loop; nothing but the error count leaves the CU):
//   bits -> 3GPP map -> IFFT -> CP                      (modem.py:797-888, ofdm.py:97-130)
//   time-variant TDL + S over the word's N data samples (fading.py:371-406)
//     + AWGN                                             (rf/noise/model.py:143-160)
//   FFT -> ideal CSI -> ZF/MMSE -> hard demap -> XOR-popcount against the bits
//     (ofdm.py:132-161, channel_estimation.py:215-295, waveform.py:235-250,
//      psk_qam_mapping.py:171-259, evaluators.py:239-258)
// Only the data windows the receiver keeps are propagated: the cyclic prefixes
// and the delay tail are discarded by the reference's demodulation
// (waveform.py:567-614) and default synchronisation (waveform.py:90-99).
#pragma once

#include <math.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "hpx_common.hpp"
#include "hpx_detect.hpp"
#include "hpx_eig.hpp"
#include "hpx_fading.hpp"
#include "hpx_fft.hpp"
#include "hpx_mapping.hpp"

namespace hpx {
int taylor_log2_block(double max_rate, int terms, int max_log2);
int ilog2_exact(int n);
}  // namespace hpx

using namespace hpx;

namespace {

constexpr int kBatchMaxThreads = 512;
constexpr int kTailPerThread = 4;  // registers holding the previous word's tail
// Complex values per thread in one FFT pass (the rows a group of the transform holds is this
// times the threads over N): by default 12 where the kernel runs in 128 registers (512 threads,
// at most 4 antennas), which keeps the FFT's registers from spilling (5 rows of 1024 points
// still form one group); 16 where registers are ample.  Heterogeneous batches may take the
// alternative instead, a tuning choice per class: 16 where the default is 12 (fewer groups,
// more registers), else 8 for 8 antennas (fewer registers, more groups) and 12 otherwise.
constexpr int fft_values_for(int nt, int maxt) { return maxt >= 512 && nt <= 4 ? 12 : 16; }
constexpr int alt_fft_values_for(int nt, int maxt) {
  return fft_values_for(nt, maxt) == 12 ? 16 : (nt == 8 ? 8 : 12);
}
template <int NT, int MAXT>
constexpr int fft_values() {
  return fft_values_for(NT, MAXT);
}
// Single-link kernels of at most 256 threads keep only the spatial realisation uniforms in a table
// (heterogeneous-batch kernels always do).
constexpr bool compact_uniforms(int maxt) { return maxt <= 256; }

struct BatchArgs {
  // link
  int n, log2n, cp, words, bps, order, detector, dc;
  int paths, sinusoids, terms, nnorm;
  int log2b, nb, dx, maxd, keep_below, xs, x0, cpl, bits_words;
  int64_t frame_len;
  double bandwidth, doppler, los_doppler, tx_scale;
  Modulation mod;
  DemapBounds dbounds;  // float32 decision boundaries of mod (exact hard decisions)
  int pad_shift;        // FFT intermediate layout: kFftPadShift, or kFftNoPad where LDS is short
  int wb;               // words simulated at once (> 1 only in the kernels of at most 256 threads)
  // arrays
  const int32_t* delays;
  const double* path_gains;
  const double* corr_rx;  // interleaved complex, may be null
  const double* corr_tx;
  const double* noise_power;
  const double* doppler_drop;  // [drop][2] NLOS, LOS Doppler, or null (the link's)
  const uint32_t* drop_index;  // [drop] Philox drop counters, or null (first_drop + drop)
  const double* normals;       // [drop][nnorm] recorded realisation normals, or null (drawn)
  int32_t* errors;
  float2* equalized;
  // frame (null elements: every element is data)
  const int32_t* elements;
  const int32_t* word_data;
  const float2* pilots;
  int nref, data_total;
  // exports, or null
  float2* out_grid;
  float2* out_csi;
  float2* out_spatial;
  uint64_t seed;
  int64_t first_drop;
  // LDS byte offsets
  int off_x, off_coef, off_abar, off_tw, off_bits, off_cons, off_s, off_det, off_red, off_dly, off_tmp_sos, off_tmp_s64;
  int off_dmb;     // the demapper's boundaries
  int off_chain;   // per path: next path of the same delay (+1, 0: none) | 1 << 16 for the first one
  // lean drops (working set beyond one CU's LDS): Taylor table and twiddles in device memory
  float2* ws_coef;
  float2* ws_tw;    // natural twiddles (the lean ideal-CSI sum)
  float2* ws_ptab;  // FFT pass table
  int off_tmp_dir;  // prologue only: per-term word-mean weights
};

// The drop kernels read their arguments through a constant-address-space pointer that goes through
// an opaque copy at every word: a field is then loaded (one scalar load, from the scalar cache) where a
// word's step uses it, instead of the ~100 fields and Philox round keys the words need being held in
// scalar registers across the loop, where most of them spilled into vector lanes and were read back one
// v_readlane each (4x4 at 1024 subcarriers: 208 spilled scalars -> 99; 4096 drops in 3.74 ms, with the words
// and segments of a drop below in the kernel, where 3.83 ms were).
#ifdef __HIP_DEVICE_COMPILE__
#define HPX_ADDRESS_SPACE(n) __attribute__((address_space(n)))
#else
#define HPX_ADDRESS_SPACE(n)  // (the host pass only parses the kernels)
#endif
typedef const HPX_ADDRESS_SPACE(4) BatchArgs ConstArgs;

// A pointer field as what it is, device memory (through a generic pointer the accesses are flat ones).
template <class T>
__device__ __forceinline__ HPX_ADDRESS_SPACE(1) T* global(T* p) {
  return (HPX_ADDRESS_SPACE(1) T*)p;
}

template <class Args>
__device__ __forceinline__ bool path_in_range(const Args& a, int p) {
  const int d = global(a.delays)[p];
  return d >= 0 && d <= a.maxd;
}

// bps bits starting at bit `bit` of an LSB-first word window (bit i of the result = i-th bit)
__device__ __forceinline__ uint32_t symbol_bits(const uint32_t* bw, int bit, int bps) {
  uint64_t v = bw[bit >> 5];
  if ((bit & 31) + bps > 32) v |= static_cast<uint64_t>(bw[(bit >> 5) + 1]) << 32;
  return static_cast<uint32_t>(v >> (bit & 31)) & ((1u << bps) - 1u);
}

// One drop, or segment seg of segs (a contiguous share of its words), simulated by the whole workgroup.
// local_drop indexes the per-drop arrays (noise power, Doppler, errors, exports); the Philox drop
// index is drop_index[local_drop] or first_drop + local_drop.  Segments of a drop add their bit errors
// to errors[local_drop], which is zero before; a drop alone (segs = 1) stores its count.
// LEAN: the segments of a drop (segs > 1) share its device workspace and only read it; a launch with
// segs = 0 before them fills it (Taylor table, twiddles, FFT pass table) and zeroes the drop's errors.
// BATCH: a.wb words go through every step at once (rows [word][stream], then the words' CSI rows), so
// that a drop of few subcarriers fills its wavefronts and takes a barrier per step and batch instead
// of per step and word.  Every value is computed by the same expression whatever the batch, the
// segment and the workgroup, so results do not depend on them.
// COMPACT: only the 100 spatial uniforms get a table, which takes up to ~8 KB off the LDS of links
// of at most 512 subcarriers, whose prologue tables bound it.  The heterogeneous-batch kernels and
// the single-link kernels of at most 256 threads take it; the 512-thread single-link kernels keep
// the full table and their code as it is (the compact form measured 5 registers more and 2.4 %
// slower on the 4x4 1024-subcarrier link).
template <int NT, int NR, int PAIRS, int FFTV, bool LEAN = false, bool COMPACT = false, bool BATCH = false>
__device__ __forceinline__ void drop_body(ConstArgs* ap, const int64_t local_drop, const int seg, const int segs) {
  extern __shared__ __align__(16) unsigned char lds[];
  ConstArgs& a = *ap;
  float2* xbuf = reinterpret_cast<float2*>(lds + a.off_x);
  // a lean drop keeps the Taylor table and the twiddles in its device workspace
  float2* coef = LEAN ? a.ws_coef : reinterpret_cast<float2*>(lds + a.off_coef);
  float2* abar = reinterpret_cast<float2*>(lds + a.off_abar);
  float2* ptab = LEAN ? a.ws_ptab : reinterpret_cast<float2*>(lds + a.off_tw);  // FFT pass table
  float2* tw = a.ws_tw;  // lean drops only: natural twiddles of the per-subcarrier ideal CSI
  uint32_t* bits = reinterpret_cast<uint32_t*>(lds + a.off_bits);
  float2* cons = reinterpret_cast<float2*>(lds + a.off_cons);
  DemapBounds* dmb = reinterpret_cast<DemapBounds*>(lds + a.off_dmb);
  float2* smat = reinterpret_cast<float2*>(lds + a.off_s);
  int* red = reinterpret_cast<int*>(lds + a.off_red);
  int* dly = reinterpret_cast<int*>(lds + a.off_dly);  // path delays: LDS broadcasts in the channel loop
  int* chain = reinterpret_cast<int*>(lds + a.off_chain);  // paths sharing a delay (ideal-CSI row)
  constexpr int kRows = NT > NR ? NT : NR;
  double* uni = reinterpret_cast<double*>(lds + a.off_x);        // prologue only
  double* sos = reinterpret_cast<double*>(lds + a.off_tmp_sos);  // prologue only
  double* s64 = reinterpret_cast<double*>(lds + a.off_tmp_s64);  // prologue only: S in float64
  double* amp_dir = reinterpret_cast<double*>(lds + a.off_tmp_dir);  // prologue only: [L][terms]
  float2* det_v = reinterpret_cast<float2*>(lds + a.off_det);     // [NT][NT] eigenvectors of S^H S
  float2* det_a = det_v + NT * NT;                                 // [NT][NR] V^H S^H
  float* det_l = reinterpret_cast<float*>(det_a + NT * NR);        // [NT] eigenvalues

  const int tid = threadIdx.x;
  const int nthreads = blockDim.x;
  const uint32_t drop = a.drop_index ? global(a.drop_index)[local_drop] : static_cast<uint32_t>(a.first_drop + local_drop);
  const int n = a.n;
  const int L = a.paths;
  const int period = n + a.cp;
  // this workgroup's words, and the Taylor blocks their windows and delays reach
  const bool tables_only = LEAN && segs == 0;
  const bool fill_tables = !LEAN || segs <= 1;
  const int parts = LEAN && segs == 0 ? 1 : segs;
  const int w_begin = static_cast<int>(static_cast<int64_t>(a.words) * seg / parts);
  const int w_end = static_cast<int>(static_cast<int64_t>(a.words) * (seg + 1) / parts);
  const int b_first = max(0, w_begin * period + a.cp - a.maxd) >> a.log2b;
  const int b_count = ((w_end * period - 1) >> a.log2b) + 1 - b_first;
  // Taylor table [path][a.nb blocks from b_first], indexed by the block itself
  float2* const coef0 = coef - (LEAN ? 0 : b_first) * kTaylorCoeffs;

  // ---------------------------------------------------------------- prologue
  // realisation uniforms Phi(z), z ~ N(0,1) (consistent.py:432,485), or z of a recorded
  // StaticConsistentRealization (consistent.py:244-260)
  if constexpr (COMPACT) {
    // Uniforms 0..99 (the spatial phases, read by several S entries) go to uni; every later one is
    // read once and goes straight into its field of the SoS table (fading.py:326-342,
    // angles/phases :492-499; rows [path][NLOS terms, then LOS] of {rate, phase, gain}): per
    // path, LOS angles, NLOS angles, LOS phases, NLOS phases, in the generator's variable order.
    const int ns = a.sinusoids, nlos = L * ns;
    const double inv_fs = 1.0 / a.bandwidth;
    const double dop = a.doppler_drop ? global(a.doppler_drop)[2 * local_drop] : a.doppler;
    const double los_dop = a.doppler_drop ? global(a.doppler_drop)[2 * local_drop + 1] : a.los_doppler;
    auto put = [&](int i, double u) {
      if (i < 100) {
        uni[i] = u;
        return;
      }
      int j = i - 100;
      if (j < L) {  // LOS angle of path j
        const double ang = 2.0 * M_PI * u;
        sos[3 * (j * a.terms + ns)] = los_dop * cos(ang) * inv_fs;
        return;
      }
      j -= L;
      if (j < nlos) {  // NLOS angle of sinusoid k of path p
        const int p = j / ns, k = j - p * ns;
        const double ang = -M_PI + 2.0 * M_PI * u;
        sos[3 * (p * a.terms + k)] = dop * cos((2.0 * M_PI * (k + 1) + ang) / ns) * inv_fs;
        return;
      }
      j -= nlos;
      if (j < L) {  // LOS phase of path j
        sos[3 * (j * a.terms + ns) + 1] = -M_PI + 2.0 * M_PI * u;
        return;
      }
      j -= L;
      const int p = j / ns, k = j - p * ns;  // NLOS phase
      sos[3 * (p * a.terms + k) + 1] = -M_PI + 2.0 * M_PI * u;
    };
    if (a.normals) {
      const auto z = global(a.normals) + local_drop * a.nnorm;
      for (int c = tid; c < a.nnorm; c += nthreads) put(c, normal_cdf(z[c]));
    } else {
      for (int c = tid; 2 * c < a.nnorm; c += nthreads) {
        const double2 z = normal_pair_f64(stream_call(a.seed, drop, HPX_STREAM_REALIZATION, static_cast<uint32_t>(c)));
        put(2 * c, normal_cdf(z.x));
        if (2 * c + 1 < a.nnorm) put(2 * c + 1, normal_cdf(z.y));
      }
    }
    for (int e = tid; e < L * a.terms; e += nthreads) {
      const int p = e / a.terms, k = e - p * a.terms;
      sos[3 * e + 2] = global(a.path_gains)[k < ns ? L + p : p];
    }
  } else {
    // all uniforms in uni; the SoS table is formed from them below
    if (a.normals) {
      const auto z = global(a.normals) + local_drop * a.nnorm;
      for (int c = tid; c < a.nnorm; c += nthreads) uni[c] = normal_cdf(z[c]);
    } else {
      for (int c = tid; 2 * c < a.nnorm; c += nthreads) {
        const double2 z = normal_pair_f64(stream_call(a.seed, drop, HPX_STREAM_REALIZATION, static_cast<uint32_t>(c)));
        uni[2 * c] = normal_cdf(z.x);
        if (2 * c + 1 < a.nnorm) uni[2 * c + 1] = normal_cdf(z.y);
      }
    }
  }
  if (tid == 0) red[0] = 0;
  // a path whose delay lies outside [0, max delay] contributes nothing: it gets delay 0 and zero
  // taps (Taylor coefficients and word means), so the channel loop needs no per-path check
  for (int p = tid; p <= L; p += nthreads) dly[p] = p < L && path_in_range(a, p) ? global(a.delays)[p] : 0;
  __syncthreads();
  // chains of paths sharing a delay, in path order: the CSI row sums their word means in the
  // order the paths are listed
  for (int p = tid; p < L; p += nthreads) {
    const int d = dly[p];
    bool first = true;
    for (int q = 0; q < p; ++q) first = first && dly[q] != d;
    int next = -1;
    for (int q = L - 1; q > p; --q)
      if (dly[q] == d) next = q;
    chain[p] = (next + 1) | (first && d < a.keep_below ? 1 << 16 : 0);
  }

  // spatial response S = R_rx exp(2 pi j U)[:NR, :NT] R_tx (fading.py:476-489)
  for (int e = tid; e < NR * NT; e += nthreads) {
    const int r = e / NT, t = e - r * NT;
    double sr = 0.0, si = 0.0;
    if (a.corr_rx) {
      for (int p = 0; p < NR; ++p)
        for (int q = 0; q < NT; ++q) {
          double s0r, s0i;
          sincospi(2.0 * uni[10 * p + q], &s0i, &s0r);
          const double ar = global(a.corr_rx)[2 * (r * NR + p)], ai = global(a.corr_rx)[2 * (r * NR + p) + 1];
          const double br = global(a.corr_tx)[2 * (q * NT + t)], bi = global(a.corr_tx)[2 * (q * NT + t) + 1];
          const double mr = ar * s0r - ai * s0i, mi = ar * s0i + ai * s0r;
          sr += mr * br - mi * bi;
          si += mr * bi + mi * br;
        }
    } else {
      sincospi(2.0 * uni[10 * r + t], &si, &sr);
    }
    smat[e] = make_float2(static_cast<float>(sr), static_cast<float>(si));
    if (a.out_spatial && seg == 0) global(a.out_spatial)[local_drop * NR * NT + e] = smat[e];
    s64[2 * e] = sr;
    s64[2 * e + 1] = si;
  }
  if constexpr (COMPACT) {
    // the word means' Dirichlet weight depends on the term only, not on the word
    for (int e = tid; e < L * a.terms; e += nthreads) amp_dir[e] = sos[3 * e + 2] * dirichlet_factor(sos[3 * e], n);
  } else {
    // SoS table (fading.py:326-342, angles/phases :492-499): NLOS terms, then LOS
    const int ns = a.sinusoids;
    const int o_los_ang = 100, o_nlos_ang = 100 + L, o_los_ph = 100 + L + L * ns, o_nlos_ph = 100 + 2 * L + L * ns;
    const double inv_fs = 1.0 / a.bandwidth;
    const double dop = a.doppler_drop ? global(a.doppler_drop)[2 * local_drop] : a.doppler;
    const double los_dop = a.doppler_drop ? global(a.doppler_drop)[2 * local_drop + 1] : a.los_doppler;
    for (int e = tid; e < L * a.terms; e += nthreads) {
      const int p = e / a.terms, k = e - p * a.terms;
      double* row = sos + 3 * e;
      if (k < ns) {
        const double ang = -M_PI + 2.0 * M_PI * uni[o_nlos_ang + p * ns + k];
        row[0] = dop * cos((2.0 * M_PI * (k + 1) + ang) / ns) * inv_fs;
        row[1] = -M_PI + 2.0 * M_PI * uni[o_nlos_ph + p * ns + k];
        row[2] = global(a.path_gains)[L + p];
      } else {
        const double ang = 2.0 * M_PI * uni[o_los_ang + p];
        row[0] = los_dop * cos(ang) * inv_fs;
        row[1] = -M_PI + 2.0 * M_PI * uni[o_los_ph + p];
        row[2] = global(a.path_gains)[p];
      }
      // the word means' Dirichlet weight depends on the term only, not on the word
      amp_dir[e] = row[2] * dirichlet_factor(row[0], n);
    }
  }
  // constellation indexed by transmitted bit order (scaled by sqrt(P_tx / N)); twiddles
  for (int v = tid; v < a.order; v += nthreads) {
    const double2 p = constellation_point(a.order, 1, bits_to_label(static_cast<uint32_t>(v), a.bps));
    cons[v] = make_float2(static_cast<float>(p.x * a.tx_scale), static_cast<float>(p.y * a.tx_scale));
  }
  if (fill_tables) fill_fft_pass_table(ptab, a.log2n);
  if (tid == 0) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      dmb->a[i] = a.dbounds.a[i];
      dmb->b[i] = a.dbounds.b[i];
    }
  }
  if (LEAN && fill_tables) {
    for (int k = tid; k < n; k += nthreads) {
      double s, c;
      sincospi(-2.0 * static_cast<double>(k) / static_cast<double>(n), &s, &c);
      tw[k] = make_float2(static_cast<float>(c), static_cast<float>(s));
    }
  }
  __syncthreads();

  // Taylor coefficients of every (path, block) and word means of every (path, word)
  const TaylorBlocks tb{a.log2b};
  // The last wavefront computes the per-drop detector of the rank-one-in-frequency ideal-CSI
  // channel on an LDS workspace while the others compute the Taylor coefficients (one
  // wavefront does both in turn).
  const bool split = nthreads >= 128;
  const int det_first = split ? nthreads - 64 : 0;
  if (tid >= det_first && !tables_only) {
    double* lam = s64 + 2 * NR * NT;
    double* v = lam + NT;
    double* am = v + 2 * NT * NT;
    spatial_detector_wave(NR, NT, s64, lam, v, am, am + 2 * NT * NR);
    const int lane = tid - det_first;
    for (int i = lane; i < NT * NT; i += 64)
      det_v[i] = make_float2(static_cast<float>(v[2 * i]), static_cast<float>(v[2 * i + 1]));
    for (int i = lane; i < NT * NR; i += 64)
      det_a[i] = make_float2(static_cast<float>(am[2 * i]), static_cast<float>(am[2 * i + 1]));
    double lmax = 0.0;
    for (int i = 0; i < NT; ++i) lmax = fmax(lmax, lam[i]);
    // numpy.linalg.pinv's cut: singular values below max(M, N) eps sigma_max are dropped
    const double rt = static_cast<double>(NR > NT ? NR : NT) * 2.220446049250313e-16;
    for (int i = lane; i < NT; i += 64) det_l[i] = lam[i] > rt * rt * lmax ? static_cast<float>(lam[i]) : 0.0f;
  }
  const int taylor_threads = split ? det_first : nthreads;
  if (tid < taylor_threads && fill_tables) {
    for (int e = tid; e < L * b_count; e += taylor_threads) {
      const int p = e / b_count, b = b_first + (e - p * b_count);
      float2* c = coef0 + (p * a.nb + b) * kTaylorCoeffs;
      if (path_in_range(a, p)) {
        taylor_coeffs(sos + 3 * p * a.terms, a.terms, tb.centre(b), tb.half_width(), c);
      } else {
#pragma unroll
        for (int k = 0; k < kTaylorCoeffs; ++k) c[k] = make_float2(0.f, 0.f);
      }
    }
  }
  if (tables_only) {
    if (tid == 0) global(a.errors)[local_drop] = 0;
    return;
  }
  for (int e = tid; e < L * (w_end - w_begin); e += nthreads) {
    const int p = e / (w_end - w_begin), w = w_begin + (e - p * (w_end - w_begin));
    abar[p * a.words + w] = path_in_range(a, p)
                                ? tap_mean_weighted(sos + 3 * p * a.terms, amp_dir + p * a.terms, a.terms,
                                                    static_cast<double>(w) * (n + a.cp) + a.cp, n)
                                : make_float2(0.f, 0.f);
  }
  __syncthreads();
  // the signal buffer aliased the prologue tables; the frame starts after silence
  for (int e = tid; e < NT * a.dx; e += nthreads) xbuf[(e / a.dx) * a.xs + (e % a.dx)] = make_float2(0.f, 0.f);

  const double np = global(a.noise_power)[local_drop];
  const float sigma = static_cast<float>(sqrt(0.5 * np));
  const float s2 = a.detector == HPX_DETECT_MMSE ? static_cast<float>(np) : 0.0f;
  const float rx_scale = static_cast<float>(1.0 / sqrt(static_cast<double>(n)));
  const int x0 = a.x0;  // LDS column of the first data sample
  int errors = 0;

  // ---------------------------------------------------------------- words
  // w: first word of a batch of nw.  A segment whose delays reach into the word before it transmits
  // that word once more (w < w_begin) for its last samples.
  const int wb = BATCH ? a.wb : 1;
  int nw = 1;
  for (int w = w_begin - (w_begin > 0 && a.dx > 0 ? 1 : 0); w < w_end; w += nw) {
    const bool lead = w < w_begin;
    if (BATCH) nw = lead ? 1 : min(wb, w_end - w);
    // e over a batch's words and elements -> word of the batch and element
    auto word_of = [&](int e, int log2) { return BATCH ? e >> log2 : 0; };
    auto elem_of = [&](int e, int log2) { return BATCH ? e & ((1 << log2) - 1) : e; };
    float2* csirow = xbuf + nw * kRows * a.xs + x0;  // [nw][xs] per-word CSI over the taps (not for lean drops)
    // The thread index passes through an opaque copy per word: the per-thread index arithmetic
    // of the word's loops is redone every word instead of being hoisted out of this loop into
    // registers held across it (which made the channel loop reload spilled values).
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    int zero;
    asm volatile("s_mov_b32 %0, 0" : "=s"(zero));
    ConstArgs& a = ap[zero];
    const uint64_t seed = a.seed;
    // bits of this word's data symbols for every stream (stream HPX_STREAM_BITS + t):
    // LSB-first words fw .. fw + nw - 1 of the stream; the word's first bit sits at bit bo
    const int wd0 = a.word_data ? global(a.word_data)[w] : w * n;
    const int wd1 = a.word_data ? global(a.word_data)[w + nw] : (w + nw) * n;
    const int64_t bit0 = static_cast<int64_t>(wd0) * a.bps;
    const int bo = static_cast<int>(bit0 & 31);
    if (wd1 > wd0) {  // (a batch whose words carry no data draws no bits)
      const int fw = static_cast<int>(bit0 >> 5);
      const int lw = static_cast<int>((static_cast<int64_t>(wd1) * a.bps - 1) >> 5);
      const int c0 = fw >> 2, c1 = lw >> 2;
      const int ncalls = c1 - c0 + 1;
      for (int e = tid; e < NT * ncalls; e += nthreads) {
        const int t = e / ncalls, c = c0 + (e - t * ncalls);
        const uint4 r = stream_call(seed, drop, HPX_STREAM_BITS + t, static_cast<uint32_t>(c));
        const uint32_t comp[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int wi = 4 * c + k - fw;
          if (wi >= 0 && wi <= lw - fw) bits[t * a.bits_words + wi] = comp[k];
        }
      }
    }
    __syncthreads();
    // map + place at the IFFT bins; clear the CSI row (row kRows: tap means at their delays)
    // (element map, bin and bit offset once per subcarrier for all streams)
    for (int e = tid; e < nw * n; e += nthreads) {
      const int wi = word_of(e, a.log2n), q = elem_of(e, a.log2n);
      const int el = a.elements ? global(a.elements)[w * n + e] : q;
      const int bin = subcarrier_bin(q, n, a.dc);
      const int wd = !BATCH ? 0 : a.word_data ? global(a.word_data)[w + wi] - wd0 : wi * n;  // data elements before the word
      const int bit = bo + (wd + el) * a.bps;
      float2* col = xbuf + wi * NT * a.xs + x0 + bin;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        float2 v;
        if (el >= 0) {
          v = cons[symbol_bits(bits + t * a.bits_words, bit, a.bps)];
        } else if (el == HPX_ELEMENT_NULL) {
          v = make_float2(0.f, 0.f);
        } else {
          const float2 pv = global(a.pilots)[t * a.nref + (-1 - el)];
          v = make_float2(static_cast<float>(static_cast<double>(pv.x) * a.tx_scale),
                          static_cast<float>(static_cast<double>(pv.y) * a.tx_scale));
        }
        col[t * a.xs] = v;
      }
      if (!LEAN) csirow[wi * a.xs + q] = make_float2(0.f, 0.f);
    }
    __syncthreads();
    lds_fft_padded<+1, FFTV, !BATCH>(xbuf + x0, nw * NT, a.xs, a.log2n, ptab, a.pad_shift);
    if (lead) {
      // only the word's last samples are wanted, as the tail of the segment's first word
      for (int e = tid; e < NT * a.dx; e += nthreads) {
        const int t = e / a.dx, i = e - t * a.dx;
        xbuf[t * a.xs + i] = xbuf[t * a.xs + x0 + n - a.dx + i];
      }
      __syncthreads();
      continue;
    }
    // cyclic prefix (only the last cpl = min(CP, max delay) prefix samples are ever read by the
    // delayed paths)
    for (int e = tid; e < nw * NT * a.cpl; e += nthreads) {
      const int t = e / a.cpl, i = e - t * a.cpl;
      xbuf[t * a.xs + x0 - a.cpl + i] = xbuf[t * a.xs + x0 + n - a.cpl + i];
    }
    // the tails of the batch's later words (the first word's was kept from the batch before)
    if (BATCH && a.dx > 0) {
      for (int e = tid; e < (nw - 1) * NT * a.dx; e += nthreads) {
        const int t = e / a.dx, i = e - t * a.dx;
        xbuf[(t + NT) * a.xs + i] = xbuf[t * a.xs + x0 + n - a.dx + i];
      }
    }
    // CSI row: word means of the taps at their delays, one thread per first path of a delay
    // (paths sharing a delay add up, taps beyond min(num_taps, N) are cut as fft(n=N) cuts them;
    // out-of-range paths have delay 0 and zero means)
    if (!LEAN) {
      for (int e = tid; e < nw * L; e += nthreads) {
        const int wi = BATCH ? e / L : 0, p = BATCH ? e - wi * L : e;
        int link = chain[p];
        if (link & (1 << 16)) {
          float2 c = abar[p * a.words + w + wi];
          for (int q = (link & 0xffff) - 1; q >= 0; q = (chain[q] & 0xffff) - 1)
            c = cadd(c, abar[q * a.words + w + wi]);
          csirow[wi * a.xs + dly[p]] = c;
        }
      }
    }
    __syncthreads();

    // channel over the data window + AWGN; y stays in registers
    const int64_t first0 = static_cast<int64_t>(w) * period + a.cp;  // absolute index of the first data sample
    float2 y[PAIRS][2][NR];
#pragma unroll
    for (int k = 0; k < PAIRS; ++k) {
      const int e = tid + k * nthreads;  // sample pair of the batch's data windows
      if (2 * e < nw * n) {
        const int wi = word_of(e, a.log2n - 1), i = elem_of(e, a.log2n - 1);
        const int nl = 2 * i;
        const int64_t win0 = first0 + (BATCH ? wi * period : 0);
        const int64_t nabs = win0 + nl;
        const float2* xrow = xbuf + (BATCH ? wi * NT * a.xs : 0) + x0 + nl;
        float2 z0[NT], z1[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) z0[t] = z1[t] = make_float2(0.f, 0.f);
        const float step = 2.0f / static_cast<float>(1 << a.log2b);  // offset of the next sample in a block
        if (first0 >= a.maxd) {
          // no delayed index reaches before the frame start: no per-lane checks
          // (the next path's delay is read one iteration ahead, off the loop's critical path)
          int d_next = dly[0];
          for (int p = 0; p < L; ++p) {
            const int d = d_next;
            d_next = dly[p + 1];
            const int m = static_cast<int>(nabs) - d;
            const int b0 = m >> a.log2b;
            // (24-bit multiply: full rate, where a 32-bit one takes four passes)
            const float2* c0 = coef0 + __umul24(static_cast<unsigned>(p * a.nb + b0), kTaylorCoeffs);
            const float s0 = tb.offset32(m);
            const float2 h0 = taylor_eval(c0, s0);
            // the pair's second sample opens the next block when m ends one
            const bool wrap = ((m + 1) >> a.log2b) != b0;
            const float2 h1 = wrap ? taylor_eval(c0 + kTaylorCoeffs, tb.offset32(m + 1)) : taylor_eval(c0, s0 + step);
            const float2* xc = xrow - d;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
              z0[t] = cfma(h0, xc[t * a.xs], z0[t]);
              z1[t] = cfma(h1, xc[t * a.xs + 1], z1[t]);
            }
          }
        } else {
          for (int p = 0; p < L; ++p) {
            const int d = dly[p];
            const int64_t m = nabs - d;
            const float2* xc = xrow - d;
            if (m >= 0) {
              const float2 h0 = taylor_eval(coef0 + (p * a.nb + static_cast<int>(tb.block_of(m))) * kTaylorCoeffs,
                                            tb.offset(m));
#pragma unroll
              for (int t = 0; t < NT; ++t) z0[t] = cfma(h0, xc[t * a.xs], z0[t]);
            }
            if (m + 1 >= 0) {
              const float2 h1 = taylor_eval(
                  coef0 + (p * a.nb + static_cast<int>(tb.block_of(m + 1))) * kTaylorCoeffs, tb.offset(m + 1));
#pragma unroll
              for (int t = 0; t < NT; ++t) z1[t] = cfma(h1, xc[t * a.xs + 1], z1[t]);
            }
          }
        }
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          float2 a0 = make_float2(0.f, 0.f), a1 = make_float2(0.f, 0.f);
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            a0 = cfma(smat[r * NT + t], z0[t], a0);
            a1 = cfma(smat[r * NT + t], z1[t], a1);
          }
          y[k][0][r] = a0;
          y[k][1][r] = a1;
        }
        // noise sample n uses words (0,1) (n even) or (2,3) (n odd) of call n/2
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          const int64_t nabs = win0 + 2 * i;
          if ((nabs & 1) == 0) {
            const uint4 wn = stream_call(seed, drop, HPX_STREAM_NOISE + r, static_cast<uint32_t>(nabs >> 1));
            const float2 n0 = complex_normal_f32(wn.x, wn.y), n1 = complex_normal_f32(wn.z, wn.w);
            y[k][0][r] = make_float2(fmaf(sigma, n0.x, y[k][0][r].x), fmaf(sigma, n0.y, y[k][0][r].y));
            y[k][1][r] = make_float2(fmaf(sigma, n1.x, y[k][1][r].x), fmaf(sigma, n1.y, y[k][1][r].y));
          } else {
            const uint4 wa = stream_call(seed, drop, HPX_STREAM_NOISE + r, static_cast<uint32_t>(nabs >> 1));
            const uint4 wb = stream_call(seed, drop, HPX_STREAM_NOISE + r, static_cast<uint32_t>((nabs + 1) >> 1));
            const float2 n0 = complex_normal_f32(wa.z, wa.w), n1 = complex_normal_f32(wb.x, wb.y);
            y[k][0][r] = make_float2(fmaf(sigma, n0.x, y[k][0][r].x), fmaf(sigma, n0.y, y[k][0][r].y));
            y[k][1][r] = make_float2(fmaf(sigma, n1.x, y[k][1][r].x), fmaf(sigma, n1.y, y[k][1][r].y));
          }
        }
      }
    }
    // last dx transmitted samples of this word feed the next word's delayed paths
    float2 tail[kTailPerThread];
#pragma unroll
    for (int k = 0; k < kTailPerThread; ++k) {
      const int e = tid + k * nthreads;
      if (e < NT * a.dx) tail[k] = xbuf[((nw - 1) * NT + e / a.dx) * a.xs + x0 + n - a.dx + (e % a.dx)];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kTailPerThread; ++k) {
      const int e = tid + k * nthreads;
      if (e < NT * a.dx) xbuf[(e / a.dx) * a.xs + (e % a.dx)] = tail[k];
    }
#pragma unroll
    for (int k = 0; k < PAIRS; ++k) {
      const int e = tid + k * nthreads;
      if (2 * e < nw * n) {
        const int wi = word_of(e, a.log2n - 1), i = elem_of(e, a.log2n - 1);
        float2* yrow = xbuf + (BATCH ? wi * NR * a.xs : 0) + x0 + 2 * i;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          yrow[r * a.xs] = y[k][0][r];
          yrow[r * a.xs + 1] = y[k][1][r];
        }
      }
    }
    __syncthreads();
    // receive FFT of every antenna and, in the same passes, the CSI row's FFT over the taps
    lds_fft_padded<-1, FFTV, !BATCH>(xbuf + x0, nw * (kRows + (LEAN ? 0 : 1)), a.xs, a.log2n, ptab, a.pad_shift);

    // ideal CSI, detection, demapping and bit errors per subcarrier
    for (int e = tid; e < nw * n; e += nthreads) {
      const int wi = word_of(e, a.log2n), q = elem_of(e, a.log2n);
      const int bin = subcarrier_bin(q, n, a.dc);
      float2 c;
      if (LEAN) {
        // the same DFT over the taps, path by path: c = sum_p abar_p W^(bin d_p)
        c = make_float2(0.f, 0.f);
        for (int p = 0; p < L; ++p) {
          const int d = dly[p];
          if (d >= 0 && d < a.keep_below) c = cfma(abar[p * a.words + w + wi], tw[(bin * d) & (n - 1)], c);
        }
      } else {
        c = csirow[wi * a.xs + bin];
      }
      // opaque zero offset: keeps the detector matrices as per-iteration LDS broadcast reads
      // instead of ~70 registers hoisted for the whole kernel
      int dofs = 0;
      asm volatile("" : "+v"(dofs));
      const float2* dva = det_v + dofs;
      const float2* daa = det_a + dofs;
      const float* dla = det_l + dofs;
      // W = V diag(conj(c) / (|c|^2 lambda_i + s2)) V^H S^H applied to y
      const float2* ycol = xbuf + (BATCH ? wi * NR * a.xs : 0) + x0 + bin;
      float2 yv[NR];
#pragma unroll
      for (int r = 0; r < NR; ++r) yv[r] = ycol[r * a.xs];
      if (a.out_grid) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
          global(a.out_grid)[((local_drop * NR + r) * a.words + w + wi) * static_cast<int64_t>(n) + q] = cscale(yv[r], rx_scale);
      }
      if (a.out_csi) global(a.out_csi)[(local_drop * a.words + w + wi) * static_cast<int64_t>(n) + q] = c;
      const int el = a.elements ? global(a.elements)[w * n + e] : q;
      if (el < 0) continue;  // reference and null elements carry no bits
      const int wd = !BATCH ? 0 : a.word_data ? global(a.word_data)[w + wi] - wd0 : wi * n;  // data elements before the word
      const float c2 = cabs2(c);
      float2 u[NT];
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        float2 acc = make_float2(0.f, 0.f);
#pragma unroll
        for (int r = 0; r < NR; ++r) acc = cfma(daa[i * NR + r], yv[r], acc);
        const float den = fmaf(c2, dla[i], s2);
        // rx_scale folds the receiver's 1/sqrt(N); a zero gain realises pinv's dropped singular values
        const float g = (dla[i] > 0.0f || s2 > 0.0f) && den > 0.0f ? rx_scale * __builtin_amdgcn_rcpf(den) : 0.0f;
        u[i] = cscale(cmulc(c, acc), g);
      }
      float2 xh[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        float2 acc = make_float2(0.f, 0.f);
#pragma unroll
        for (int i = 0; i < NT; ++i) acc = cfma(dva[t * NT + i], u[i], acc);
        xh[t] = acc;
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const uint32_t rx = demap_symbol_f32(a.mod.pam, dmb, xh[t].x, xh[t].y);
        const uint32_t tx = symbol_bits(bits + t * a.bits_words, bo + (wd + el) * a.bps, a.bps);
        errors += __popc(tx ^ rx);
        if (a.equalized) global(a.equalized)[(local_drop * NT + t) * static_cast<int64_t>(a.data_total) + wd0 + wd + el] = xh[t];
      }
    }
    __syncthreads();
  }

  // ---------------------------------------------------------------- epilogue
  for (int off = 32; off > 0; off >>= 1) errors += __shfl_down(errors, off, 64);
  if ((tid & 63) == 0) atomicAdd(red, errors);
  __syncthreads();
  if (tid == 0) {
    if (segs == 1) global(a.errors)[local_drop] = red[0];
    else if (red[0]) __hip_atomic_fetch_add(global(a.errors) + local_drop, red[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Wavefronts per SIMD the registers are kept for.  512-thread workgroups: 4 (128 VGPRs, two drops per CU)
// for the 4x4 link of up to 1024 subcarriers, which its LDS allows, measured 1.6x faster than 256
// VGPRs at one drop per CU; 6 (three drops per CU) for one and two antennas; 2 where the LDS holds one
// drop (4x4 beyond 1024 subcarriers, 8x8).
template <int NT, int PAIRS, int MAXT>
constexpr int batch_waves_per_eu() {
  return NT == 8 ? 2 : MAXT < 512 ? 4 : NT == 4 ? (PAIRS == 1 ? 4 : 2) : PAIRS == 1 ? 6 : 4;
}

template <int NT, int NR, int PAIRS, int MAXT, bool BATCH = false>
__global__ void __launch_bounds__(MAXT) __attribute__((amdgpu_waves_per_eu(batch_waves_per_eu<NT, PAIRS, MAXT>())))
batch_kernel(BatchArgs a, int segs, int first) {
  const int drop = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x) / segs);
  // (the arguments where they lie: a is the kernel's first parameter)
  drop_body<NT, NR, PAIRS, fft_values<NT, MAXT>(), false, compact_uniforms(MAXT), BATCH>(
      (ConstArgs*)__builtin_amdgcn_kernarg_segment_ptr(), first + drop, static_cast<int>(blockIdx.x) - drop * segs, segs);
}

// Heterogeneous batches: workgroup i simulates the drop plans[i] describes; its first_drop is
// the drop's Philox index and its per-drop pointers already point at the drop's entries.
template <int NT, int NR, int PAIRS, int MAXT, bool LEAN = false, int FFTV = fft_values<NT, MAXT>(), bool BATCH = false>
__global__ void __launch_bounds__(MAXT) __attribute__((amdgpu_waves_per_eu(batch_waves_per_eu<NT, PAIRS, MAXT>())))
batch_kernel_multi(const BatchArgs* __restrict__ plans, int segs) {
  const int parts = LEAN && segs == 0 ? 1 : segs;
  const int slot = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x) / parts);
  const int seg = static_cast<int>(blockIdx.x) - slot * parts;
  // a drop of fewer steps than the launch has segments makes one segment a step; the others would only repeat its prologue
  ConstArgs* plan = (ConstArgs*)(plans + slot);
  if (segs > 1) {
    const int most = (plan->words + plan->wb - 1) / plan->wb;
    if (seg >= most) return;
    segs = min(segs, most);
  }
  drop_body<NT, NR, PAIRS, FFTV, LEAN, true, BATCH>(plan, 0, seg, segs);
}

// Zero error counts of drops whose segments add to them (a kernel, so that a captured graph holds no
// memset node).
__global__ void __launch_bounds__(256) zero_errors_kernel(int32_t* errors, int count) {
  const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < count) errors[i] = 0;
}
__global__ void __launch_bounds__(256) zero_plan_errors_kernel(const BatchArgs* __restrict__ plans, int count) {
  const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < count) plans[i].errors[0] = 0;
}

// Workgroup size of kernels that run several words side by side: 256 threads, 128 at 8 antennas, whose
// registers allow two wavefronts per SIMD (four drops per CU instead of two).  6400 drops of 15 paths at 64,
// 128 and 256 threads: 1x1 at 64 subcarriers 712, 480, 396 us, 4x4 at 128 subcarriers 1828, 1083, 937 us,
// 8x8 at 128 subcarriers 3122, 2251, 2937 us.
constexpr int kBatchThreads = 256;
constexpr int batch_threads(int nt) { return nt <= 4 ? kBatchThreads : 128; }
// Heterogeneous classes of fewer threads and one sample pair per thread run so.
constexpr bool batched_class(int nt, int threads, int pairs) { return threads < batch_threads(nt) && pairs == 1; }

constexpr int64_t kMaxLds = 160 * 1024;

inline int64_t align16(int64_t v) { return (v + 15) & ~int64_t(15); }

// Wavefronts per CU a kernel's registers allow (512 VGPRs per SIMD lane in steps of 8, at most 8 wavefronts).
inline int waves_per_cu(const void* fn) {
  hipFuncAttributes attr;
  if (hipFuncGetAttributes(&attr, fn) != hipSuccess || attr.numRegs <= 0) return 8;
  return 4 * std::min(8, 512 / ((attr.numRegs + 7) & ~7));
}

// Drops of `threads` threads each in one launch, which holds fewer than 2^32.
inline int64_t drops_per_launch(int threads) { return 0xffffffffll / threads; }

inline int device_cus() {
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess)
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 256;
  return cus;
}

// Workgroups a CU holds at once, by LDS and by registers.
inline int64_t workgroups_per_cu(int cu_waves, int threads, int64_t lds) {
  const int64_t by_waves = static_cast<int64_t>(cu_waves) * 64 / threads;
  return std::max<int64_t>(1, std::min<int64_t>(kMaxLds / std::max<int64_t>(lds, 1), by_waves));
}

// Workgroups a drop's words are spread over.  The drops of a small launch leave much of the GPU idle
// while each steps through its words, and a launch of a little more than the GPU holds leaves it
// idle in its second round, so a drop is cut into the segments for which a launch is shortest: rounds of
// the GPU times what a segment takes, its prologue and its steps.  A segment repeats the prologue, whatever the
// frame's length, and a part of the word before it where delays reach into it, and a launch that zeroes the
// errors goes before.  A full GPU slows prologue and steps, so the last round costs less the emptier it is.
// Times in word steps, of 10 us (1x1 at 64 subcarriers) to 35 us (8x8 at 1024), from launches of 1 to 20000 drops of 1 to
// 40 words: of 916 such shapes of 32 to 1024 subcarriers and 1 to 8 antennas the choice is slower than whole drops of
// N / 2 threads by at most 5 %, and 1.65 times as fast in the mean.  One drop of 64 subcarriers 131 -> 31 us, one 4x4 drop of
// 1024 subcarriers 355 -> 63 us, 1000 2x2 drops of 512 subcarriers with exports 586 -> 441 us; 700 4x4 drops of 1024
// subcarriers and 3 words stay whole, 165 us, 216 in two segments.
constexpr double kLead = 0.35, kZero = 0.3;
constexpr double kStepFull = 0.36;  // what a full GPU adds to a step

// A workgroup's prologue, what a full GPU adds to it, and a step of its threads.
struct GroupTimes {
  double prologue, prologue_full, step;
};
inline GroupTimes group_times(int nt, int threads, bool batch) {
  const double one = nt == 1 ? 2.3 : nt == 2 ? 2.0 : 1.6;  // (the detector of more antennas hides behind the rest)
  // one wavefront does the detector after the rest, and waits for each step alone
  if (threads <= 64) return {one + (nt == 1 ? 0.2 : nt == 2 ? 0.4 : 0.6), 0.5, nt == 8 ? 1.0 : batch ? 1.25 : 1.1};
  return threads <= 128 ? GroupTimes{one + 0.1, 0.36, 1.0} : GroupTimes{one, 0.28, threads <= 256 ? 0.9 : 1.0};
}
// Time of a launch of `groups` workgroups of `steps` steps of which the GPU holds `resident`.
inline double launch_time(const GroupTimes& g, int64_t groups, int64_t resident, double steps) {
  const int64_t rounds = groups / resident;
  const double rest = static_cast<double>(groups - rounds * resident) / static_cast<double>(resident);
  auto in_rounds = [&](double full) { return static_cast<double>(rounds) * (1.0 + full) + (rest > 0.0 ? 1.0 + full * rest : 0.0); };
  return g.prologue * in_rounds(g.prologue_full) + steps * g.step * in_rounds(kStepFull);
}
struct Segments {
  int count = 1;
  double time = 0.0;  // of the launch
};
// steps(s): steps of the longest of s segments; resident(s): segments the GPU holds
template <class Steps, class Resident>
Segments segments_for(const GroupTimes& g, int64_t drops, int most, double lead, Steps steps, Resident resident) {
  Segments best;
  for (int s = 1; s <= most; ++s) {
    const double t = launch_time(g, drops * s, resident(s), steps(s) + (s > 1 ? lead : 0.0)) + (s > 1 ? kZero : 0.0);
    if (s == 1 || t < best.time) best = {s, t};
  }
  return best;
}
// Heterogeneous classes: their words per drop are known to the plans only (a drop makes no more segments than it has
// steps), and they share the GPU with the classes of other streams, so a class's segments fill at most half of it.  Lean
// drops, one of which a CU holds and which take 1.5 ms each in one piece, are cut too, after a launch that fills
// their workspaces.  Mixed batches of 64, 300, 1000, 2048 and 8192 drops on four streams: whole 2754, 3970, 3591, 3678 and
// 8211 us, in segments that may fill the GPU 660, 897, 1600, 2893 and 8587, half of it 671, 894, 1584, 2736 and
// 8247; of 3 words each instead of 14, 2048 and 8192 drops 1021 and 2172, 1260 and 2448, 922 and 2156.
constexpr int kMultiMaxSegments = 7;
constexpr double kMultiWords = 14.0;  // a drop's steps, for the rule's sake

// Raises a kernel's dynamic LDS limit once per process and size (so that launches recorded
// into a graph after a first eager run make no attribute calls).
bool ensure_lds(const void* fn, int64_t bytes) {
  static std::mutex mu;
  static std::map<const void*, int64_t> granted;
  if (bytes <= 64 * 1024) return true;
  std::lock_guard<std::mutex> lock(mu);
  int64_t& g = granted[fn];
  if (g >= bytes) return true;
  if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)) != hipSuccess)
    return false;
  g = bytes;
  return true;
}

template <int NT, int MAXT, bool LEAN, int FFTV>
int launch_multi_kernel(const BatchArgs* plans, const hpx_uneven_class& c, hipStream_t stream) {
  void (*fn)(const BatchArgs*, int) = nullptr;
  switch (c.pairs) {
    case 1: fn = batch_kernel_multi<NT, NT, 1, MAXT, LEAN, FFTV>; break;
    case 2: fn = batch_kernel_multi<NT, NT, 2, MAXT, LEAN, FFTV>; break;
    case 4: fn = batch_kernel_multi<NT, NT, 4, MAXT, LEAN, FFTV>; break;
    default: set_error("hpx_uneven_run: unsupported samples per thread"); return HPX_ERR_UNSUPPORTED;
  }
  if constexpr (MAXT <= kBatchThreads && !LEAN) {
    if (batched_class(NT, c.threads, c.pairs)) fn = batch_kernel_multi<NT, NT, 1, MAXT, LEAN, FFTV, true>;
  }
  if (!ensure_lds(reinterpret_cast<const void*>(fn), c.lds_bytes)) {
    set_error("hpx_uneven_run: %lld bytes of LDS per workgroup not available", static_cast<long long>(c.lds_bytes));
    return HPX_ERR_UNSUPPORTED;
  }
  const BatchArgs* const all = plans + c.first;
  const int threads = batched_class(NT, c.threads, c.pairs) ? batch_threads(NT) : c.threads;
  const int64_t resident =
      device_cus() * workgroups_per_cu(waves_per_cu(reinterpret_cast<const void*>(fn)), threads, c.lds_bytes);
  const int most = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(kMultiMaxSegments, resident / (2 * c.count))));
  const int segs = segments_for(group_times(NT, threads, threads > c.threads), c.count, most, 0.0,
                                [](int s) { return kMultiWords / s; }, [&](int) { return resident; }).count;
  const int64_t pieces = drops_per_launch(threads * segs);
  for (int64_t at = 0; at < c.count; at += pieces) {
    const BatchArgs* const first = all + at;
    const int64_t count = std::min(pieces, c.count - at);
    if (LEAN && segs > 1)  // the workspaces first
      hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>(count)), dim3(threads), c.lds_bytes, stream, first, 0);
    else if (segs > 1)
      hipLaunchKernelGGL(zero_plan_errors_kernel, dim3(static_cast<unsigned>((count + 255) / 256)), dim3(256), 0, stream,
                         first, static_cast<int>(count));
    hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>(count * segs)), dim3(threads), c.lds_bytes, stream, first, segs);
  }
  return check_launch("hpx_uneven_run");
}

// One class launch with the FFT values per thread `fftv` (lean classes exist only for 8x8 links,
// the one shape beyond one CU's LDS).
template <int NT, int MAXT, int FFTV>
int launch_multi_fftv(const BatchArgs* plans, const hpx_uneven_class& c, hipStream_t stream) {
  if constexpr (NT == 8) {
    if (c.lean) return launch_multi_kernel<NT, MAXT, true, FFTV>(plans, c, stream);
  }
  if (c.lean) {
    set_error("hpx_uneven_run: lean class with %d antennas", NT);
    return HPX_ERR_INVALID;
  }
  return launch_multi_kernel<NT, MAXT, false, FFTV>(plans, c, stream);
}

struct Plan {
  int threads = 0, pairs = 0;  // threads per word, sample pairs per thread
  int launch_threads = 0;      // workgroup size
  int antennas = 0;
  int segs = 1;                // segments per drop (single-link launches)
  bool batch = false;          // several words side by side
  int fftv = 0;  // FFT values per thread and pass
  int64_t lds = 0;
  bool lean = false;      // Taylor table and twiddles in device memory, ideal CSI per subcarrier
  int64_t ws_elems = 0;   // complex64 workspace elements of a lean drop
  BatchArgs args{};
};

// Blocks of a segment's Taylor table, of its own words only, and the bytes of a table.
inline int segment_blocks(const BatchArgs& a, int segs) {
  if (segs == 1) return a.nb;
  const int64_t period = a.n + a.cp;
  const int64_t span = (a.words + segs - 1) / segs * period + std::max(0, a.maxd - a.cp);
  return static_cast<int>(std::min<int64_t>(a.nb, ((span - 2) >> a.log2b) + 2));
}
inline int64_t table_bytes(const BatchArgs& a, int nb) {
  return align16(static_cast<int64_t>(a.paths) * nb * kTaylorCoeffs * sizeof(float2));
}

// Segments of a single-link launch on `cus` CUs whose registers allow cu_waves wavefronts each.
inline Segments plan_segments(const Plan& plan, int64_t num_drops, int cu_waves, int cus) {
  const BatchArgs& a = plan.args;
  // a thread's second sample pair nearly doubles a step (1x1 at 256 subcarriers on 64 threads)
  const double step = a.n > 2 * plan.launch_threads ? 0.95 * a.n / (2 * plan.launch_threads) : 1.0;
  return segments_for(
      group_times(plan.antennas, plan.launch_threads, plan.batch), num_drops, (a.words + a.wb - 1) / a.wb, a.dx > 0 ? kLead : 0.0,
      [&](int s) { return step * (((a.words + s - 1) / s + a.wb - 1) / a.wb); },
      [&](int s) {
        const int64_t lds = plan.lds - table_bytes(a, a.nb) + table_bytes(a, segment_blocks(a, s));
        return cus * workgroups_per_cu(cu_waves, plan.launch_threads, lds);
      });
}

// Cuts the drops of a single-link launch: the shorter Taylor table shortens the LDS layout after it.
inline void set_segments(Plan* plan, int segs) {
  if (segs == 1) return;
  BatchArgs& a = plan->args;
  plan->segs = segs;
  const int nb = segment_blocks(a, segs);
  const int less = static_cast<int>(table_bytes(a, a.nb) - table_bytes(a, nb));
  a.nb = nb;
  plan->lds -= less;
  for (int* off : {&a.off_abar, &a.off_tw, &a.off_bits, &a.off_cons, &a.off_s, &a.off_det, &a.off_red, &a.off_dly, &a.off_dmb,
                   &a.off_chain})
    *off -= less;
}

template <class K>
int launch(K kernel, Plan plan, int64_t num_drops, hipStream_t stream) {
  set_segments(&plan, plan_segments(plan, num_drops, waves_per_cu(reinterpret_cast<const void*>(kernel)), device_cus()).count);
  if (!ensure_lds(reinterpret_cast<const void*>(kernel), plan.lds)) {
    set_error("hpx_run_batch: %lld bytes of LDS per workgroup not available", static_cast<long long>(plan.lds));
    return HPX_ERR_UNSUPPORTED;
  }
  if (plan.segs > 1)
    hipLaunchKernelGGL(zero_errors_kernel, dim3(static_cast<unsigned>((num_drops + 255) / 256)), dim3(256), 0, stream,
                       plan.args.errors, static_cast<int>(num_drops));
  const int64_t most = drops_per_launch(plan.launch_threads * plan.segs);
  for (int64_t first = 0; first < num_drops; first += most)
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(std::min(most, num_drops - first) * plan.segs)),
                       dim3(plan.launch_threads), plan.lds, stream, plan.args, plan.segs, static_cast<int>(first));
  return check_launch("hpx_run_batch");
}

template <int NT, int MAXT>
int launch_pairs(const Plan& plan, int64_t num_drops, hipStream_t stream) {
  if constexpr (MAXT <= kBatchThreads) {
    if (plan.batch) return launch(batch_kernel<NT, NT, 1, MAXT, true>, plan, num_drops, stream);
  }
  switch (plan.pairs) {
    case 1: return launch(batch_kernel<NT, NT, 1, MAXT>, plan, num_drops, stream);
    case 2: return launch(batch_kernel<NT, NT, 2, MAXT>, plan, num_drops, stream);
    case 4: return launch(batch_kernel<NT, NT, 4, MAXT>, plan, num_drops, stream);
  }
  set_error("hpx_run_batch: unsupported samples per thread");
  return HPX_ERR_UNSUPPORTED;
}

// One class launch with the default or the alternative FFT values per thread.
template <int NT, bool ALT>
int launch_multi(const BatchArgs* plans, const hpx_uneven_class& c, hipStream_t stream) {
  constexpr int big = ALT ? alt_fft_values_for(NT, 512) : fft_values_for(NT, 512);
  constexpr int small = ALT ? alt_fft_values_for(NT, 256) : fft_values_for(NT, 256);
  return c.threads > 256 ? launch_multi_fftv<NT, 512, big>(plans, c, stream)
                         : launch_multi_fftv<NT, 256, small>(plans, c, stream);
}

template <int NT>
int launch_single(const Plan& plan, int64_t num_drops, hipStream_t stream) {
  return plan.launch_threads <= 256 ? launch_pairs<NT, 256>(plan, num_drops, stream)
                                    : launch_pairs<NT, 512>(plan, num_drops, stream);
}

}  // namespace
