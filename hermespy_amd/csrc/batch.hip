// Fused Monte Carlo link drops: host side (validation, launch plans, heterogeneous batches) and the
// float64 single-antenna drops.  The kernels are in hpx_drop.hpp.
#include "hpx_drop.hpp"

// Launchers, one translation unit per antenna count and kind (batch_<antennas>.hip, batch_alt_<antennas>.hip).
#define HPX_DECLARE_LAUNCHERS(NT)                                                                        \
  int batch_launch_single_##NT(const void* plan, int64_t num_drops, hipStream_t s);                      \
  int batch_launch_multi_##NT(const void* plans_dev, const hpx_uneven_class& c, hipStream_t s);          \
  int batch_launch_alt_##NT(const void* plans_dev, const hpx_uneven_class& c, hipStream_t s);
namespace hpx {
HPX_DECLARE_LAUNCHERS(1)
HPX_DECLARE_LAUNCHERS(2)
HPX_DECLARE_LAUNCHERS(4)
HPX_DECLARE_LAUNCHERS(8)
}  // namespace hpx
#undef HPX_DECLARE_LAUNCHERS

namespace {

constexpr int64_t kBatchLds = 52 * 1024;  // batches of words: at least three drops per CU

// LDS layout of a plan; a lean layout leaves out the Taylor table, the FFT pass table and the
// CSI row.  pad: rows long enough for the FFT's padded intermediate layout (N + N / 8 after the
// first data sample).
int64_t layout_lds(BatchArgs& a, int nr, int nt, bool lean, bool pad, bool compact) {
  const int rows = a.wb * (std::max(nr, nt) + (lean ? 0 : 1));  // signal rows (+ the CSI row) of a batch's words
  a.pad_shift = pad ? kFftPadShift : kFftNoPad;
  a.xs = a.x0 + a.n + (pad ? (a.n >> kFftPadShift) : 0);
  a.xs += a.xs & 1;
  int64_t o = 0;
  a.off_x = 0;
  const int64_t xbytes = static_cast<int64_t>(rows) * a.xs * sizeof(float2);
  const int64_t uni_bytes = align16(static_cast<int64_t>(compact ? std::min(a.nnorm, 100) : a.nnorm) * sizeof(double));
  const int64_t sos_bytes = align16(static_cast<int64_t>(a.paths) * a.terms * 3 * sizeof(double));
  // S (float64), then the detector's outputs and Jacobi workspace
  const int64_t s64_bytes =
      static_cast<int64_t>(2 * nr * nt + nt + 2 * nt * nt + 2 * nt * nr + kEigWork) * sizeof(double);
  const int64_t s64_aligned = align16(s64_bytes);
  const int64_t dir_bytes = align16(static_cast<int64_t>(a.paths) * a.terms * sizeof(double));
  o += align16(std::max(xbytes, uni_bytes + sos_bytes + s64_aligned + dir_bytes));
  a.off_tmp_sos = static_cast<int>(uni_bytes);
  a.off_tmp_s64 = static_cast<int>(uni_bytes + sos_bytes);
  a.off_tmp_dir = static_cast<int>(uni_bytes + sos_bytes + s64_aligned);
  a.off_coef = static_cast<int>(o);
  if (!lean) o += align16(static_cast<int64_t>(a.paths) * a.nb * kTaylorCoeffs * sizeof(float2));
  a.off_abar = static_cast<int>(o);
  o += align16(static_cast<int64_t>(a.paths) * a.words * sizeof(float2));
  a.off_tw = static_cast<int>(o);
  if (!lean) o += align16(static_cast<int64_t>(a.n) * sizeof(float2));
  a.off_bits = static_cast<int>(o);
  o += align16(static_cast<int64_t>(nt) * a.bits_words * sizeof(uint32_t));
  a.off_cons = static_cast<int>(o);
  o += align16(static_cast<int64_t>(a.order) * sizeof(float2));
  a.off_s = static_cast<int>(o);
  o += align16(static_cast<int64_t>(nr) * nt * sizeof(float2));
  a.off_det = static_cast<int>(o);
  o += align16(static_cast<int64_t>(nt * nt + nt * nr) * sizeof(float2) + nt * sizeof(float));
  a.off_red = static_cast<int>(o);
  o += 16;
  a.off_dly = static_cast<int>(o);
  o += align16(static_cast<int64_t>(a.paths + 1) * sizeof(int32_t));  // + a pad entry for the prefetch
  a.off_dmb = static_cast<int>(o);
  o += align16(sizeof(DemapBounds));
  a.off_chain = static_cast<int>(o);
  o += align16(static_cast<int64_t>(a.paths) * sizeof(int32_t));
  return o;
}

// Validates the link (and frame, if any) and computes the launch geometry and LDS layout.
// allow_lean: an 8x8 link beyond one CU's LDS gets the lean layout (heterogeneous batches,
// which provide its workspace).
// exact_taps: the caller evaluates every tap sample directly (the float64 path), so no Taylor
// block size bounds the Doppler rate.
int make_plan(const hpx_link* l, const hpx_frame* f, Plan* out, bool allow_lean = false, bool exact_taps = false) {
  HPX_REQUIRE(l, "hpx_run_batch: null link");
  if (f) {
    HPX_REQUIRE(f->elements && f->word_data, "hpx_run_batch_frames: null frame arrays");
    HPX_REQUIRE(f->num_references >= 0 && (f->num_references == 0 || f->pilots),
                "hpx_run_batch_frames: reference elements need pilot symbols");
    HPX_REQUIRE(f->num_data >= 0 && f->max_word_data >= 0 && f->max_word_data <= l->num_subcarriers,
                "hpx_run_batch_frames: invalid data element counts");
  }
  const int log2n = ilog2_exact(l->num_subcarriers);
  if (log2n < 5 || l->num_subcarriers > 4096) {
    set_error("hpx_run_batch: num_subcarriers must be a power of two in [32, 4096] (got %d)", l->num_subcarriers);
    return HPX_ERR_UNSUPPORTED;
  }
  HPX_REQUIRE(l->words >= 1 && l->prefix >= 0 && l->prefix <= l->num_subcarriers, "hpx_run_batch: invalid frame");
  HPX_REQUIRE(l->num_paths >= 1 && l->num_sinusoids >= 1 && l->max_delay >= 0,
              "hpx_run_batch: invalid path configuration");
  HPX_REQUIRE(l->bandwidth > 0.0, "hpx_run_batch: bandwidth must be positive");
  HPX_REQUIRE(l->device_power >= 0.0, "hpx_run_batch: device power must be non-negative");
  HPX_REQUIRE(l->detector == HPX_DETECT_ZF || l->detector == HPX_DETECT_MMSE, "hpx_run_batch: unknown detector");
  const bool known = l->num_tx == 1 || l->num_tx == 2 || l->num_tx == 4 || l->num_tx == 8;
  if (l->num_rx != l->num_tx || !known) {
    set_error("hpx_run_batch: antenna configuration %dx%d not instantiated (1x1, 2x2, 4x4, 8x8)", l->num_rx,
              l->num_tx);
    return HPX_ERR_UNSUPPORTED;
  }
  Modulation mod;
  if (l->modulation_order == 2 || !modulation(l->modulation_order, 1, &mod)) {
    set_error("hpx_run_batch: modulation order %d not supported (4, 16, 64, 256)", l->modulation_order);
    return HPX_ERR_UNSUPPORTED;
  }
  BatchArgs& a = out->args;
  a.n = l->num_subcarriers;
  a.log2n = log2n;
  a.cp = l->prefix;
  a.words = l->words;
  a.bps = mod.bps;
  a.order = l->modulation_order;
  a.mod = mod;
  a.dbounds = demap_bounds_of(mod);
  a.detector = l->detector;
  a.dc = l->dc_suppression ? 1 : 0;
  a.paths = l->num_paths;
  a.sinusoids = l->num_sinusoids;
  a.terms = l->num_sinusoids + 1;
  a.nnorm = 100 + 2 * l->num_paths + 2 * l->num_paths * l->num_sinusoids;
  a.frame_len = static_cast<int64_t>(l->words) * (l->num_subcarriers + l->prefix);
  a.bandwidth = l->bandwidth;
  a.doppler = l->doppler;
  a.los_doppler = l->los_doppler;
  a.tx_scale = sqrt(l->device_power) / sqrt(static_cast<double>(l->num_subcarriers));
  const double max_rate = std::max(fabs(l->doppler), fabs(l->los_doppler)) / l->bandwidth;
  a.log2b = taylor_log2_block(max_rate, a.terms, 11);
  if (exact_taps) a.log2b = std::max(a.log2b, 6);
  if (a.log2b < 6) {
    set_error("hpx_run_batch: Doppler rate %.3g rad/sample too high for the block Taylor taps", max_rate);
    return HPX_ERR_UNSUPPORTED;
  }
  a.nb = static_cast<int>((a.frame_len + (int64_t(1) << a.log2b) - 1) >> a.log2b);
  const int max_word_data = f ? f->max_word_data : l->num_subcarriers;
  a.data_total = f ? f->num_data : l->words * l->num_subcarriers;
  a.nref = f ? f->num_references : 0;
  a.maxd = l->max_delay;
  a.dx = std::max(0, l->max_delay - a.cp);
  if (a.dx > a.n) {
    set_error("hpx_run_batch: delay spread of %d samples exceeds one OFDM word", l->max_delay);
    return HPX_ERR_UNSUPPORTED;
  }
  // LDS row: [previous word's last dx samples | last min(CP, D) prefix samples | N data samples
  // (| the FFT's padding)]; the row stride a.xs is set with the layout
  a.cpl = std::min(a.cp, l->max_delay);
  a.x0 = a.dx + a.cpl;  // == max delay
  a.keep_below = static_cast<int>(std::min<int64_t>(std::min<int64_t>(1 + l->max_delay, a.frame_len), a.n));

  const int nt = l->num_tx, nr = l->num_rx;
  int threads = std::min(kBatchMaxThreads, std::max(64, l->num_subcarriers / 2));
  if (l->workgroup_size != 0) {
    const int w = l->workgroup_size;
    if (w < 64 || w > kBatchMaxThreads || (w & (w - 1))) {
      set_error("hpx_run_batch: workgroup_size must be 0 or a power of two in [64, %d]", kBatchMaxThreads);
      return HPX_ERR_INVALID;
    }
    threads = w;
  }
  const int pairs = std::max(1, l->num_subcarriers / (2 * threads));
  if (pairs != 1 && pairs != 2 && pairs != 4) {
    set_error("hpx_run_batch: %d subcarriers need %d sample pairs per thread at %d threads (1, 2 or 4)",
              l->num_subcarriers, pairs, threads);
    return HPX_ERR_UNSUPPORTED;
  }
  if (l->num_subcarriers > kFftMaxPerThread * threads) {
    set_error("hpx_run_batch: %d subcarriers exceed one workgroup's FFT capacity", l->num_subcarriers);
    return HPX_ERR_UNSUPPORTED;
  }
  if (nt * a.dx > kTailPerThread * threads) {
    set_error("hpx_run_batch: inter-word delay tail too long (%d samples)", a.dx);
    return HPX_ERR_UNSUPPORTED;
  }
  out->threads = threads;
  out->pairs = pairs;
  out->antennas = nt;
  {
    const int maxt = threads <= 256 ? 256 : 512;
    const int def = fft_values_for(nt, maxt), alt = alt_fft_values_for(nt, maxt);
    if (l->fft_values != 0 && l->fft_values != def && l->fft_values != alt) {
      set_error("hpx_run_batch: fft_values must be 0, %d or %d for %d antennas at %d threads (got %d)", def, alt, nt,
                threads, l->fft_values);
      return HPX_ERR_INVALID;
    }
    out->fftv = l->fft_values != 0 ? l->fft_values : def;
  }

  // Words side by side: heterogeneous batches do so for the classes batched_class() names, single links
  // wherever a word's sample pairs leave threads of the workgroup idle; the default workgroup of links
  // of few subcarriers is made for it.
  const bool multi_batch = allow_lean && batched_class(nt, threads, pairs);
  const int lt = multi_batch || (!allow_lean && l->workgroup_size == 0) ? std::max(threads, batch_threads(nt)) : threads;
  out->launch_threads = lt;
  out->batch = lt <= kBatchThreads && pairs == 1 && (allow_lean ? multi_batch : 2 * lt > l->num_subcarriers);
  // LDS layout; the prologue tables (uniforms, SoS table) alias the signal buffer.  The FFT's
  // padded layout is taken where it keeps as many drops per CU as the plain one.
  auto set_words = [&](int wb) {
    a.wb = wb;
    // a batch's data bits start anywhere in an LSB-first 32-bit word
    a.bits_words = (wb * max_word_data * mod.bps + 63) >> 5;
  };
  set_words(1);
  auto per_cu = [&](int64_t bytes) {
    const int64_t by_waves = static_cast<int64_t>(lt >= 512 ? (nt <= 4 ? 4 : 2) : 4) * 4 * 64 / lt;
    return bytes > kMaxLds ? int64_t(0) : std::min<int64_t>(kMaxLds / bytes, std::max<int64_t>(1, by_waves));
  };
  auto best_layout = [&](bool lean) {
    BatchArgs padded = a;
    // the kernel these threads launch: heterogeneous batches (allow_lean) always take the compact form
    const bool compact = allow_lean || compact_uniforms(threads <= 256 ? 256 : 512);
    const int64_t op = layout_lds(padded, nr, nt, lean, true, compact);
    const int64_t on = layout_lds(a, nr, nt, lean, false, compact);
    if (per_cu(op) >= per_cu(on) && op <= kMaxLds) {
      a = padded;
      return op;
    }
    return on;
  };
  int64_t o = best_layout(false);
  if (out->batch && o <= kMaxLds) {
    // as many words as the workgroup's sample pairs hold, evenly shared over the batches of the frame,
    // while the rows stay within kBatchLds (or what one word takes)
    const int64_t one = o;
    for (int most = std::min(l->words, lt * 2 / l->num_subcarriers); most > 1; --most) {
      set_words((l->words + (l->words + most - 1) / most - 1) / ((l->words + most - 1) / most));
      o = best_layout(false);
      if (o <= std::max<int64_t>(one, kBatchLds)) break;
      most = a.wb;
      set_words(1);
      o = best_layout(false);
    }
  }
  if (o > kMaxLds && allow_lean && nt == 8) {
    o = best_layout(true);
    out->lean = true;
    // [Taylor table | natural twiddles | FFT pass table]
    out->ws_elems = static_cast<int64_t>(a.paths) * a.nb * kTaylorCoeffs + a.n + fft_pass_table_size(a.n);
  }
  out->lds = o;
  if (o > kMaxLds) {
    set_error("hpx_run_batch: link needs %lld bytes of LDS per drop (max 163840)", static_cast<long long>(o));
    return HPX_ERR_UNSUPPORTED;
  }
  return HPX_OK;
}

}  // namespace

extern "C" int64_t hpx_uneven_workspace_elements(const hpx_link* link_host) {
  if (!link_host) {
    set_error("hpx_uneven_workspace_elements: null pointer");
    return -1;
  }
  Plan plan;
  if (make_plan(link_host, nullptr, &plan, true) != HPX_OK) return -1;
  return plan.lean ? plan.ws_elems : 0;
}

extern "C" int64_t hpx_uneven_plan_bytes(void) { return static_cast<int64_t>(sizeof(BatchArgs)); }

namespace {

// Plans of a heterogeneous batch.  Lean drops take their workspace from tables_host[i].workspace,
// or, with scratch_base set, consecutive slices of scratch_base (scratch_elems complex64 values).
int uneven_prepare(const hpx_link* links_host, const hpx_drop_tables* tables_host, const uint32_t* drop_index_host,
                   int64_t num_drops, uint64_t seed, const double* noise_power, int32_t* errors, void* plans_host,
                   int64_t* order_host, hpx_uneven_class* classes_host, int max_classes, int* num_classes_host,
                   float2* scratch_base, int64_t scratch_elems) {
  HPX_REQUIRE(num_drops >= 0 && num_drops <= 0x7fffffff && max_classes >= 1, "hpx_uneven_prepare: invalid sizes");
  HPX_REQUIRE(num_classes_host, "hpx_uneven_prepare: null pointer");
  *num_classes_host = 0;
  if (num_drops == 0) return HPX_OK;
  HPX_REQUIRE(links_host && tables_host && drop_index_host && noise_power && errors && plans_host && order_host &&
                  classes_host,
              "hpx_uneven_prepare: null pointer");
  std::vector<Plan> plans(static_cast<size_t>(num_drops));
  int64_t scratch_used = 0;
  for (int64_t i = 0; i < num_drops; ++i) {
    const hpx_drop_tables& tb = tables_host[i];
    HPX_REQUIRE(tb.delays && tb.path_gains, "hpx_uneven_prepare: drop %lld has no path tables",
                static_cast<long long>(i));
    HPX_REQUIRE((tb.corr_rx == nullptr) == (tb.corr_tx == nullptr),
                "hpx_uneven_prepare: give both correlation matrices or none");
    const int st = make_plan(&links_host[i], nullptr, &plans[i], true);
    if (st != HPX_OK) return st;
    BatchArgs& a = plans[i].args;
    if (plans[i].lean) {
      float2* ws = reinterpret_cast<float2*>(tb.workspace);
      if (scratch_base) {
        if (scratch_used + plans[i].ws_elems > scratch_elems) {
          set_error("hpx_uneven_prepare_noalloc: the lean drops need more than the %lld complex64 values of the "
                    "library's scratch array",
                    static_cast<long long>(scratch_elems));
          return HPX_ERR_INVALID;
        }
        ws = scratch_base + scratch_used;
        scratch_used += plans[i].ws_elems;
      }
      HPX_REQUIRE(ws, "hpx_uneven_prepare: drop %lld needs a workspace of %lld elements", static_cast<long long>(i),
                  static_cast<long long>(plans[i].ws_elems));
      a.ws_coef = ws;
      a.ws_tw = ws + static_cast<int64_t>(a.paths) * a.nb * kTaylorCoeffs;
      a.ws_ptab = a.ws_tw + a.n;
    }
    a.delays = tb.delays;
    a.path_gains = tb.path_gains;
    a.equalized = reinterpret_cast<float2*>(tb.equalized);
    a.corr_rx = reinterpret_cast<const double*>(tb.corr_rx);
    a.corr_tx = reinterpret_cast<const double*>(tb.corr_tx);
    a.noise_power = noise_power + i;
    a.errors = errors + i;
    a.seed = seed;
    a.first_drop = drop_index_host[i];
  }
  // kernel class = (antennas, threads, samples per thread, lean, FFT values per thread), split by
  // subcarrier count so that a class holds one link shape (which a tuner times per shape; with
  // the default workgroup sizes the kernel already determines it); heavier classes and drops first
  auto key = [&](int64_t i) {
    return std::make_tuple(links_host[i].num_tx, plans[i].threads, plans[i].pairs, plans[i].lean ? 1 : 0,
                           plans[i].fftv, links_host[i].num_subcarriers);
  };
  auto cost = [&](int64_t i) {
    const hpx_link& l = links_host[i];
    return static_cast<double>(l.num_tx) * l.num_rx * l.words * (l.num_subcarriers + l.prefix) * l.num_paths;
  };
  std::vector<int64_t> idx(static_cast<size_t>(num_drops));
  for (int64_t i = 0; i < num_drops; ++i) idx[i] = i;
  std::map<std::tuple<int, int, int, int, int, int>, double> class_cost;
  for (int64_t i = 0; i < num_drops; ++i) class_cost[key(i)] = std::max(class_cost[key(i)], cost(i));
  std::stable_sort(idx.begin(), idx.end(), [&](int64_t x, int64_t y) {
    const auto kx = key(x), ky = key(y);
    if (kx != ky) {
      const double cx = class_cost[kx], cy = class_cost[ky];
      return cx != cy ? cx > cy : kx < ky;
    }
    return cost(x) > cost(y);
  });
  BatchArgs* out = static_cast<BatchArgs*>(plans_host);
  int nc = 0;
  for (int64_t k = 0; k < num_drops; ++k) {
    const int64_t i = idx[k];
    out[k] = plans[i].args;
    order_host[k] = i;
    const bool fresh = k == 0 || key(idx[k - 1]) != key(i);
    if (fresh) {
      if (nc == max_classes) {
        set_error("hpx_uneven_prepare: more than %d kernel classes", max_classes);
        return HPX_ERR_INVALID;
      }
      hpx_uneven_class& c = classes_host[nc++];
      c.first = k;
      c.count = 0;
      c.num_tx = links_host[i].num_tx;
      c.threads = plans[i].threads;
      c.pairs = plans[i].pairs;
      c.lean = plans[i].lean ? 1 : 0;
      c.lds_bytes = 0;
      c.fft_values = plans[i].fftv;
      c.reserved = 0;
    }
    hpx_uneven_class& c = classes_host[nc - 1];
    c.count += 1;
    c.lds_bytes = std::max<int64_t>(c.lds_bytes, plans[i].lds);
  }
  *num_classes_host = nc;
  return HPX_OK;
}

}  // namespace

// Scratch of hpx_uneven_prepare_noalloc: lean drops' Taylor and twiddle tables.  Each device holds
// its own copy until the process ends; host code never uses the name itself, only the address
// hipGetSymbolAddress gives for the current device.
constexpr int64_t kNoAllocScratchElems = int64_t(1) << 22;  // complex64 values: 32 MiB
static __device__ __align__(256) float scratch[2 * kNoAllocScratchElems];

namespace {

constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxScratchDevices] = {};

// The current device's address of `scratch`, looked up once per device.
int scratch_address(float2** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxScratchDevices) {
    set_error("hpx_uneven_prepare_noalloc: no current HIP device");
    return HPX_ERR_DEVICE;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      set_error("hpx_uneven_prepare_noalloc: hipGetSymbolAddress: %s", hipGetErrorString(e));
      return HPX_ERR_DEVICE;
    }
    g_scratch_ptr[dev] = p;
  }
  *out = static_cast<float2*>(g_scratch_ptr[dev]);
  return HPX_OK;
}

}  // namespace

extern "C" int hpx_uneven_prepare(const hpx_link* links_host, const hpx_drop_tables* tables_host,
                                  const uint32_t* drop_index_host, int64_t num_drops, uint64_t seed,
                                  const double* noise_power, int32_t* errors, void* plans_host, int64_t* order_host,
                                  hpx_uneven_class* classes_host, int max_classes, int* num_classes_host) {
  return uneven_prepare(links_host, tables_host, drop_index_host, num_drops, seed, noise_power, errors, plans_host,
                        order_host, classes_host, max_classes, num_classes_host, nullptr, 0);
}

extern "C" int64_t hpx_uneven_noalloc_capacity(void) { return kNoAllocScratchElems; }

extern "C" int hpx_uneven_prepare_noalloc(const hpx_link* links_host, const hpx_drop_tables* tables_host,
                                          const uint32_t* drop_index_host, int64_t num_drops, uint64_t seed,
                                          const double* noise_power, int32_t* errors, void* plans_host,
                                          int64_t* order_host, hpx_uneven_class* classes_host, int max_classes,
                                          int* num_classes_host) {
  int64_t need = 0;
  if (links_host && num_drops > 0) {
    for (int64_t i = 0; i < num_drops; ++i) {
      Plan p;
      if (make_plan(&links_host[i], nullptr, &p, true) == HPX_OK && p.lean) need += p.ws_elems;
    }
  }
  if (need > kNoAllocScratchElems) {
    set_error("hpx_uneven_prepare_noalloc: the lean drops need %lld complex64 values of workspace, the library's "
              "scratch array holds %lld",
              static_cast<long long>(need), static_cast<long long>(kNoAllocScratchElems));
    return HPX_ERR_INVALID;
  }
  float2* base = nullptr;
  if (need > 0) {
    const int st = scratch_address(&base);
    if (st != HPX_OK) return st;
  }
  return uneven_prepare(links_host, tables_host, drop_index_host, num_drops, seed, noise_power, errors, plans_host,
                        order_host, classes_host, max_classes, num_classes_host, base, kNoAllocScratchElems);
}

extern "C" int hpx_uneven_run(const void* plans, const hpx_uneven_class* classes_host, int num_classes,
                              void* stream) {
  HPX_REQUIRE(num_classes >= 0, "hpx_uneven_run: invalid class count");
  if (num_classes == 0) return HPX_OK;
  HPX_REQUIRE(plans && classes_host, "hpx_uneven_run: null pointer");
  const hipStream_t s = static_cast<hipStream_t>(stream);
  for (int k = 0; k < num_classes; ++k) {
    const hpx_uneven_class& c = classes_host[k];
    HPX_REQUIRE(c.count >= 0 && c.count <= 0x7fffffff && c.first >= 0, "hpx_uneven_run: invalid class");
    if (c.count == 0) continue;
    const int maxt = c.threads > 256 ? 512 : 256;
    const bool alt = c.fft_values != fft_values_for(c.num_tx, maxt);
    if (alt && c.fft_values != alt_fft_values_for(c.num_tx, maxt)) {
      set_error("hpx_uneven_run: %d FFT values per thread not available for %d antennas at %d threads", c.fft_values,
                c.num_tx, c.threads);
      return HPX_ERR_INVALID;
    }
    int st = HPX_ERR_UNSUPPORTED;
    switch (c.num_tx) {
      case 1: st = alt ? hpx::batch_launch_alt_1(plans, c, s) : hpx::batch_launch_multi_1(plans, c, s); break;
      case 2: st = alt ? hpx::batch_launch_alt_2(plans, c, s) : hpx::batch_launch_multi_2(plans, c, s); break;
      case 4: st = alt ? hpx::batch_launch_alt_4(plans, c, s) : hpx::batch_launch_multi_4(plans, c, s); break;
      case 8: st = alt ? hpx::batch_launch_alt_8(plans, c, s) : hpx::batch_launch_multi_8(plans, c, s); break;
      default: set_error("hpx_uneven_run: antenna count %d not instantiated", c.num_tx);
    }
    if (st != HPX_OK) return st;
  }
  return HPX_OK;
}

extern "C" int64_t hpx_run_batch_lds_bytes(const hpx_link* link_host) {
  Plan plan;
  if (make_plan(link_host, nullptr, &plan) != HPX_OK) return 0;
  return plan.lds;
}

extern "C" int hpx_run_batch(const hpx_link* link_host, const int32_t* delays, const double* path_gains,
                             const hpx_c128* corr_rx, const hpx_c128* corr_tx, uint64_t seed, int64_t first_drop,
                             int64_t num_drops, const double* noise_power, int32_t* errors, hpx_c64* equalized,
                             void* stream) {
  hpx_batch_out out{};
  out.errors = errors;
  out.equalized = equalized;
  return hpx_run_batch_frames(link_host, nullptr, delays, path_gains, corr_rx, corr_tx, nullptr, seed, first_drop,
                              num_drops, noise_power, &out, stream);
}

extern "C" int hpx_run_batch_frames(const hpx_link* link_host, const hpx_frame* frame_host, const int32_t* delays,
                                    const double* path_gains, const hpx_c128* corr_rx, const hpx_c128* corr_tx,
                                    const double* doppler, uint64_t seed, int64_t first_drop, int64_t num_drops,
                                    const double* noise_power, const hpx_batch_out* out_host, void* stream) {
  hpx_drop_inputs in{};
  in.noise_power = noise_power;
  in.doppler = doppler;
  return hpx_run_batch_drops(link_host, frame_host, delays, path_gains, corr_rx, corr_tx, &in, seed, first_drop,
                             num_drops, out_host, stream);
}

extern "C" int hpx_run_batch_drops(const hpx_link* link_host, const hpx_frame* frame_host, const int32_t* delays,
                                   const double* path_gains, const hpx_c128* corr_rx, const hpx_c128* corr_tx,
                                   const hpx_drop_inputs* in_host, uint64_t seed, int64_t first_drop,
                                   int64_t num_drops, const hpx_batch_out* out_host, void* stream) {
  HPX_REQUIRE(out_host && in_host, "hpx_run_batch: null input or output descriptor");
  int32_t* errors = out_host->errors;
  const double* noise_power = in_host->noise_power;
  const double* doppler = in_host->doppler;
  HPX_REQUIRE(delays && path_gains && noise_power && errors, "hpx_run_batch: null pointer");
  HPX_REQUIRE((corr_rx == nullptr) == (corr_tx == nullptr), "hpx_run_batch: give both correlation matrices or none");
  HPX_REQUIRE(num_drops >= 0 && num_drops <= 0x7fffffff, "hpx_run_batch: invalid drop count");
  HPX_REQUIRE(in_host->drop_index || (first_drop >= 0 && first_drop + num_drops <= (int64_t(1) << 32)),
              "hpx_run_batch: drop index exceeds 32 bits");
  Plan plan;
  const int st = make_plan(link_host, frame_host, &plan);
  if (st != HPX_OK) return st;
  if (plan.fftv != fft_values_for(link_host->num_tx, plan.launch_threads <= 256 ? 256 : 512)) {
    set_error("hpx_run_batch: the alternative FFT values per thread apply to heterogeneous batches only");
    return HPX_ERR_UNSUPPORTED;
  }
  if (num_drops == 0) return HPX_OK;
  if (link_host->workgroup_size == 0 && link_host->num_subcarriers <= 2 * kBatchThreads) {
    // Workgroups of 64 to batch_threads() threads, words side by side where that leaves threads idle: large ones take
    // fewer steps over a drop's words, small ones leave the GPU room for more drops, whose prologues hardly
    // gain from threads.  The shorter launch by the model of segments_for; of drops that fill the GPU the
    // one-word workgroup (N / 2 threads) unless another wins clearly.  1x1, 6 paths, 64, 128 and 256 threads: 128 subcarriers and one word, 20000
    // drops 255, 366 and 597 us, 2000 drops 43, 43 and 70; 14 words, 20000 drops 1450, 1242 and 1426 us, 700 drops
    // 96, 89 and 79; 256 subcarriers and 3 words, 20000 drops 506, 612 and 834 us.
    const int cus = device_cus(), waves = link_host->num_tx == 8 ? 8 : 16;
    const int one_word = std::max(64, link_host->num_subcarriers / 2);
    const bool full = num_drops > cus * workgroups_per_cu(waves, plan.launch_threads, plan.lds);
    auto time_of = [&](const Plan& p) {
      return plan_segments(p, num_drops, waves, cus).time * (full && p.launch_threads == one_word ? 0.9 : 1.0);
    };
    double best = time_of(plan);
    const int made = plan.launch_threads;
    for (int t = 64; t <= batch_threads(link_host->num_tx); t *= 2) {
      if (t == made || link_host->num_subcarriers > 4 * t) continue;
      hpx_link other = *link_host;
      other.workgroup_size = t;
      Plan p;
      if (make_plan(&other, frame_host, &p) != HPX_OK) continue;
      const double time = time_of(p);
      if (time < best) {
        best = time;
        plan = p;
      }
    }
  }
  BatchArgs& a = plan.args;
  a.delays = delays;
  a.path_gains = path_gains;
  a.corr_rx = reinterpret_cast<const double*>(corr_rx);
  a.corr_tx = reinterpret_cast<const double*>(corr_tx);
  a.noise_power = noise_power;
  a.errors = errors;
  a.equalized = reinterpret_cast<float2*>(out_host->equalized);
  a.doppler_drop = doppler;
  a.drop_index = in_host->drop_index;
  a.normals = in_host->normals;
  a.elements = frame_host ? frame_host->elements : nullptr;
  a.word_data = frame_host ? frame_host->word_data : nullptr;
  a.pilots = frame_host ? reinterpret_cast<const float2*>(frame_host->pilots) : nullptr;
  a.out_grid = reinterpret_cast<float2*>(out_host->grid);
  a.out_csi = reinterpret_cast<float2*>(out_host->csi);
  a.out_spatial = reinterpret_cast<float2*>(out_host->spatial);
  a.seed = seed;
  a.first_drop = first_drop;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  switch (link_host->num_tx) {
    case 1: return hpx::batch_launch_single_1(&plan, num_drops, s);
    case 2: return hpx::batch_launch_single_2(&plan, num_drops, s);
    case 4: return hpx::batch_launch_single_4(&plan, num_drops, s);
    case 8: return hpx::batch_launch_single_8(&plan, num_drops, s);
  }
  set_error("hpx_run_batch: unreachable antenna configuration");
  return HPX_ERR_UNSUPPORTED;
}

// ---------------------------------------------------------------- float64 single-antenna drops
// The float64 counterpart of the fused drop for single-antenna links of up to 256 subcarriers:
// the same counter-based streams and the same steps, every value a double, the taps summed
// exactly over their sinusoids at every sample (fading.py:293-343) instead of from Taylor blocks.
// One 256-thread workgroup per drop, all words of the frame at once.
//
// Bound: float64 VALU issue.  A sinusoid at output sample n = 64 Q + 8 a + b of a path of delay d is
// the product of three table entries, A e^{j phi} e^{j w (64 Q - d)}, e^{j 8 w a} and e^{j w b}: per
// path (frame / 64 + 16) x terms sines and cosines instead of frame x terms, and per 8 samples and
// term one complex product and 8 multiply-adds on table entries that LDS broadcasts.  Every phase
// is a product w x samples near zero, which costs less rounding than a direct evaluation's
// w x samples + phi, and the products add about as much back: the error is about the same.  The OFDM transforms are radix-4 Stockham passes over the whole
// frame between the two signal buffers (less rounding than the direct sums they replace).  The
// tables and the prologue's uniforms live in the receive buffer, which is empty until the channel's
// outputs leave their registers, so four drops share a CU.  5000 drops of 64 subcarriers, 5 paths:
// 2398 us with a sine and cosine per sample and direct sums, 478 us now.
namespace {

constexpr int kF64Threads = 256;
constexpr int kF64MaxSubcarriers = 256;
constexpr int kF64Run = 8;       // consecutive output samples per thread
constexpr int kF64Block = 64;    // samples per first factor of the phase
constexpr int kF64Round = kF64Run * kF64Threads;  // output samples per round of the workgroup
constexpr int kF64Tables = 512;  // complex128 values the tables may take beyond a short frame's

struct F64Layout {
  int off_sos, off_tw, off_x, off_y, off_abar, off_bits, off_red;
  int dx, frame, bits_words;
  int work;        // complex128 values of the receive buffer: the frame, or more for the sinusoids' tables
  int term_group;  // sinusoids whose tables fit the receive buffer at once
  int64_t bytes;
};

__device__ __forceinline__ double2 dcmul(double2 a, double2 b) {
  return make_double2(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ double2 dcfma(double2 a, double2 b, double2 c) {
  return make_double2(fma(a.x, b.x, fma(-a.y, b.y, c.x)), fma(a.x, b.y, fma(a.y, b.x, c.y)));
}
__device__ __forceinline__ double2 dcadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 dcsub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }

// One Stockham pass of radix R (4 or 2) of `rows` N-point vectors, vector v from src + v sstride to
// dst + v dstride; with prefix > 0 the outputs k >= N - prefix are also stored N samples earlier (the
// cyclic prefix).  tw[k] = exp(-2 pi j k / N); SIGN = +1 conjugates it.
template <int SIGN, int R>
__device__ __forceinline__ void f64_fft_pass(const double2* src, int sstride, double2* dst, int dstride, int rows,
                                             int log2n, int log2ns, const double2* tw, int prefix) {
  constexpr int kLog2R = R == 4 ? 2 : 1;
  const int n = 1 << log2n, log2nr = log2n - kLog2R, nr = 1 << log2nr, ns = 1 << log2ns;
  for (int item = threadIdx.x; item < rows << log2nr; item += kF64Threads) {
    const int v = item >> log2nr, j = item & (nr - 1), pos = j & (ns - 1);
    const int step = pos << (log2n - log2ns - kLog2R);
    double2 a[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
      a[k] = src[v * sstride + j + k * nr];
      if (k && ns > 1) {
        const double2 t = tw[k * step];
        a[k] = dcmul(a[k], make_double2(t.x, SIGN < 0 ? t.y : -t.y));
      }
    }
    if constexpr (R == 4) {
      const double2 t0 = dcadd(a[0], a[2]), t1 = dcsub(a[0], a[2]), t2 = dcadd(a[1], a[3]), t3 = dcsub(a[1], a[3]);
      const double2 t3j = SIGN < 0 ? make_double2(t3.y, -t3.x) : make_double2(-t3.y, t3.x);
      a[0] = dcadd(t0, t2);
      a[1] = dcadd(t1, t3j);
      a[2] = dcsub(t0, t2);
      a[3] = dcsub(t1, t3j);
    } else {
      const double2 t = a[0];
      a[0] = dcadd(t, a[1]);
      a[1] = dcsub(t, a[1]);
    }
    const int o = ((j - pos) << kLog2R) + pos;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int k = o + r * ns;
      dst[v * dstride + k] = a[r];
      if (k >= n - prefix) dst[v * dstride + k - n] = a[r];
    }
  }
  __syncthreads();
}

__device__ __forceinline__ int f64_fft_passes(int log2n) { return (log2n + 1) >> 1; }

// All passes of `rows` transforms: from src (stride sstride) alternately to b (stride N) and a (stride N),
// the last pass to last (stride lstride), which must not be the buffer it reads.
template <int SIGN>
__device__ __forceinline__ void f64_fft(const double2* src, int sstride, double2* a, double2* b, double2* last, int lstride,
                                        int rows, int log2n, const double2* tw, int prefix) {
  const int n = 1 << log2n, passes = f64_fft_passes(log2n);
  int log2ns = 0;
  for (int p = 0; p < passes; ++p) {
    double2* dst = p == passes - 1 ? last : (p & 1 ? a : b);
    const int ds = p == passes - 1 ? lstride : n, pre = p == passes - 1 ? prefix : 0;
    if (log2n - log2ns >= 2) f64_fft_pass<SIGN, 4>(src, sstride, dst, ds, rows, log2n, log2ns, tw, pre);
    else f64_fft_pass<SIGN, 2>(src, sstride, dst, ds, rows, log2n, log2ns, tw, pre);
    log2ns += 2;
    src = dst;
    sstride = ds;
  }
}

// RUN: output samples per thread of the channel, consecutive: kF64Run, or one for frames of at most a workgroup's threads,
// whose few runs of eight would be one long chain (the same products and sums per sample): one drop of a word of 32
// subcarriers and 15 paths 119 us in runs of eight, 59 in single samples, 109 with a sine and cosine per sample.
template <int RUN>
__global__ void __launch_bounds__(kF64Threads) __attribute__((amdgpu_waves_per_eu(4)))
f64_drop_kernel(BatchArgs a, F64Layout g, double2* equalized) {
  extern __shared__ __align__(16) unsigned char lds[];
  double* sos = reinterpret_cast<double*>(lds + g.off_sos);
  double2* tw = reinterpret_cast<double2*>(lds + g.off_tw);    // [N] exp(-2 pi j k / N)
  double2* x = reinterpret_cast<double2*>(lds + g.off_x);      // [dx + frame] transmitted, dx leading zeros
  double2* y = reinterpret_cast<double2*>(lds + g.off_y);      // [frame] received
  double2* abar = reinterpret_cast<double2*>(lds + g.off_abar);  // [L][words] word means of the taps
  uint32_t* bits = reinterpret_cast<uint32_t*>(lds + g.off_bits);
  int* red = reinterpret_cast<int*>(lds + g.off_red);
  double* uni = reinterpret_cast<double*>(x);       // prologue only
  double* dir = reinterpret_cast<double*>(y);       // prologue only: [L][terms] word-mean weights
  const int tid = threadIdx.x;
  const int64_t local_drop = blockIdx.x;
  const uint32_t drop = static_cast<uint32_t>(a.first_drop + local_drop);
  const int n = a.n, L = a.paths, period = a.n + a.cp, terms = a.terms;

  // realisation uniforms, the data bits (stream HPX_STREAM_BITS, LSB first), twiddles
  for (int c = tid; 2 * c < a.nnorm; c += kF64Threads) {
    const double2 z = normal_pair_f64(stream_call(a.seed, drop, HPX_STREAM_REALIZATION, static_cast<uint32_t>(c)));
    uni[2 * c] = normal_cdf(z.x);
    if (2 * c + 1 < a.nnorm) uni[2 * c + 1] = normal_cdf(z.y);
  }
  for (int c = tid; 4 * c < g.bits_words; c += kF64Threads) {
    const uint4 r = stream_call(a.seed, drop, HPX_STREAM_BITS, static_cast<uint32_t>(c));
    const uint32_t comp[4] = {r.x, r.y, r.z, r.w};
    for (int k = 0; k < 4 && 4 * c + k < g.bits_words; ++k) bits[4 * c + k] = comp[k];
  }
  for (int k = tid; k < n; k += kF64Threads) {
    double s, c;
    sincospi(-2.0 * static_cast<double>(k) / static_cast<double>(n), &s, &c);
    tw[k] = make_double2(c, s);
  }
  if (tid == 0) red[0] = 0;
  __syncthreads();

  // SoS table (fading.py:326-342, :492-499): per term the rate and A e^{j phi}, so that every later
  // phase is a product rate x samples near zero, which rounds far less than rate x samples + phi
  {
    const int ns = a.sinusoids;
    const int o_los_ang = 100, o_nlos_ang = 100 + L, o_los_ph = 100 + L + L * ns, o_nlos_ph = 100 + 2 * L + L * ns;
    const double inv_fs = 1.0 / a.bandwidth;
    for (int e = tid; e < L * terms; e += kF64Threads) {
      const int p = e / terms, k = e - p * terms;
      double rate, phase, amp;
      if (k < ns) {
        const double ang = -M_PI + 2.0 * M_PI * uni[o_nlos_ang + p * ns + k];
        rate = a.doppler * cos((2.0 * M_PI * (k + 1) + ang) / ns) * inv_fs;
        phase = -M_PI + 2.0 * M_PI * uni[o_nlos_ph + p * ns + k];
        amp = a.path_gains[L + p];
      } else {
        const double ang = 2.0 * M_PI * uni[o_los_ang + p];
        rate = a.los_doppler * cos(ang) * inv_fs;
        phase = -M_PI + 2.0 * M_PI * uni[o_los_ph + p];
        amp = a.path_gains[p];
      }
      double sn, cs;
      sincos(phase, &sn, &cs);
      double* row = sos + 3 * e;
      row[0] = rate;
      row[1] = amp * cs;
      row[2] = amp * sn;
      if (e < g.work * 2) dir[e] = dirichlet_factor(rate, n);
    }
  }
  // spatial response of the single antenna pair: exp(2 pi j u_00) (fading.py:476-489)
  double2 S;
  sincospi(2.0 * uni[0], &S.y, &S.x);
  __syncthreads();
  // word means (the Dirichlet closed form): four lanes per (path, word), each every fourth sinusoid
  for (int e0 = 0; e0 < 4 * L * a.words; e0 += kF64Threads) {
    const int e = (e0 + tid) >> 2;
    double ar = 0.0, ai = 0.0;
    if (e < L * a.words) {
      const int p = e / a.words, w = e - p * a.words;
      if (path_in_range(a, p)) {
        const double centre = static_cast<double>(w) * period + a.cp + 0.5 * static_cast<double>(n - 1);
        for (int k = tid & 3; k < terms; k += 4) {
          const int i = p * terms + k;
          const double rate = sos[3 * i];
          const double wgt = i < g.work * 2 ? dir[i] : dirichlet_factor(rate, n);
          double s, c;
          sincos(reduce_phase(rate * centre), &s, &c);
          const double2 v = dcmul(make_double2(sos[3 * i + 1], sos[3 * i + 2]), make_double2(c, s));
          ar = fma(wgt, v.x, ar);
          ai = fma(wgt, v.y, ai);
        }
      }
    }
    ar += __shfl_xor(ar, 1, 64);
    ai += __shfl_xor(ai, 1, 64);
    ar += __shfl_xor(ar, 2, 64);
    ai += __shfl_xor(ai, 2, 64);
    if (e < L * a.words && (tid & 3) == 0) abar[e] = make_double2(ar, ai);
  }
  __syncthreads();

  // transmit: map every word's symbols, inverse DFTs (unnormalised, the constellation carries
  // sqrt(P / N)), prefixes; the last pass goes to x, so an even number of passes starts there
  {
    double2* xd = x + g.dx;
    const bool even = (f64_fft_passes(a.log2n) & 1) == 0;
    double2* sym = even ? xd : y;
    for (int e = tid; e < a.words << a.log2n; e += kF64Threads) {
      const int w = e >> a.log2n, q = e & (n - 1);
      const uint32_t v = symbol_bits(bits, e * a.bps, a.bps);
      const double2 p = constellation_point(a.order, 1, bits_to_label(v, a.bps));
      sym[(w << a.log2n) + subcarrier_bin(q, n, a.dc)] = make_double2(p.x * a.tx_scale, p.y * a.tx_scale);
    }
    __syncthreads();
    f64_fft<+1>(sym, n, even ? xd : y, even ? y : xd, xd + a.cp, period, a.words, a.log2n, tw, a.cp);
    for (int i = tid; i < g.dx; i += kF64Threads) x[i] = make_double2(0.0, 0.0);
    __syncthreads();
  }

  // channel: y_n = S sum_l h_l(n - d_l) x_(n - d_l) + sqrt(P / 2) (N + jN) over the frame, a round of
  // kF64Round samples at a time from the end of the frame (the tables lie at the start of y)
  const double np = a.noise_power[local_drop];
  const double sigma = sqrt(0.5 * np);
  for (int r0 = (g.frame - 1) / kF64Round * kF64Round; r0 >= 0; r0 -= kF64Round) {
    const int blocks = (min(kF64Round, g.frame - r0) + kF64Block - 1) / kF64Block;
    const int n0 = r0 + RUN * tid;
    const bool active = n0 < g.frame;
    double2 z[RUN];
#pragma unroll
    for (int b = 0; b < RUN; ++b) z[b] = make_double2(0.0, 0.0);
    for (int p = 0; p < L; ++p) {
      if (!path_in_range(a, p)) continue;
      const int d = a.delays[p];
      double2 h[RUN];
#pragma unroll
      for (int b = 0; b < RUN; ++b) h[b] = make_double2(0.0, 0.0);
      for (int t0 = 0; t0 < terms; t0 += g.term_group) {
        const int tg = min(g.term_group, terms - t0);
        // tables [tg][blocks | 8 | 8]
        const int row = blocks + 2 * kF64Run;
        __syncthreads();
        for (int e = tid; e < tg * row; e += kF64Threads) {
          const int k = e / row, c = e - k * row;
          const double* sp = sos + 3 * (p * terms + t0 + k);
          const int m = c < blocks ? r0 + c * kF64Block - d
                        : c < blocks + kF64Run ? (c - blocks) * kF64Run : c - blocks - kF64Run;
          double sn, cs;
          sincos(reduce_phase(sp[0] * static_cast<double>(m)), &sn, &cs);
          const double2 v = make_double2(cs, sn);
          y[e] = c < blocks ? dcmul(make_double2(sp[1], sp[2]), v) : v;
        }
        __syncthreads();
        if (active) {
          const double2* tq = y + (n0 - r0) / kF64Block;
          const double2* ta = y + blocks + ((n0 / kF64Run) & (kF64Block / kF64Run - 1));
          const double2* tb = y + blocks + kF64Run + (n0 & (kF64Run - 1));
          for (int k = 0; k < tg; ++k) {
            const double2 c = dcmul(tq[k * row], ta[k * row]);
#pragma unroll
            for (int b = 0; b < RUN; ++b) h[b] = dcfma(c, tb[k * row + b], h[b]);
          }
        }
      }
      if (active) {
#pragma unroll
        for (int b = 0; b < RUN; ++b) {
          const int m = n0 + b - d;  // (x holds dx >= d zeros before the frame)
          if (n0 + b < g.frame) z[b] = dcfma(h[b], x[g.dx + m], z[b]);
        }
      }
    }
    __syncthreads();
    if (active) {
#pragma unroll
      for (int b = 0; b < RUN; b += 2) {
        // noise sample i: words (0, 1) of call i / 2 for even i, (2, 3) for odd i
        const uint4 wn = stream_call(a.seed, drop, HPX_STREAM_NOISE, static_cast<uint32_t>((n0 + b) >> 1));
#pragma unroll
        for (int j = 0; j < (RUN > 1 ? 2 : 1); ++j) {
          const int i = n0 + b + j, o = RUN > 1 ? j : i & 1;
          if (i >= g.frame) break;
          const uint32_t w0 = o ? wn.z : wn.x, w1 = o ? wn.w : wn.y;
          const double u1 = (static_cast<double>(w0 >> 8) + 0.5) * 5.9604644775390625e-08;
          const double u2 = static_cast<double>(w1 >> 8) * 5.9604644775390625e-08;
          const double rho = sigma * sqrt(-2.0 * log(u1));
          double ns, nc;
          sincospi(2.0 * u2, &ns, &nc);
          const double2 v = dcmul(S, z[b + j]);
          y[i] = make_double2(fma(rho, nc, v.x), fma(rho, ns, v.y));
        }
      }
    }
  }
  __syncthreads();

  // receive: DFTs of the words' data windows, ideal CSI, ZF / MMSE, demap, bit errors
  const bool odd = (f64_fft_passes(a.log2n) & 1) != 0;
  double2* spec = odd ? x : y;
  f64_fft<-1>(y + a.cp, period, y, x, spec, n, a.words, a.log2n, tw, 0);
  const double rx_scale = 1.0 / sqrt(static_cast<double>(n));
  const double s2 = a.detector == HPX_DETECT_MMSE ? np : 0.0;
  int errors = 0;
  for (int e = tid; e < a.words << a.log2n; e += kF64Threads) {
    const int w = e >> a.log2n, q = e & (n - 1);
    const int bin = subcarrier_bin(q, n, a.dc);
    const double2 yv = spec[(w << a.log2n) + bin];
    const double yr = yv.x * rx_scale, yi = yv.y * rx_scale;
    double2 c = make_double2(0.0, 0.0);
    for (int p = 0; p < L; ++p) {
      const int d = a.delays[p];
      if (!path_in_range(a, p) || d >= a.keep_below) continue;
      c = dcfma(abar[p * a.words + w], tw[(bin * d) & (n - 1)], c);
    }
    const double hr = S.x * c.x - S.y * c.y, hi = S.x * c.y + S.y * c.x;
    const double den = hr * hr + hi * hi + s2;
    const double gain = den > 0.0 ? 1.0 / den : 0.0;  // pinv of a zero channel is zero
    const double xr = (hr * yr + hi * yi) * gain, xi = (hr * yi - hi * yr) * gain;
    const uint32_t rx = demap_symbol(a.mod, xr, xi);
    const uint32_t tx = symbol_bits(bits, e * a.bps, a.bps);
    errors += __popc(tx ^ rx);
    if (equalized) equalized[local_drop * static_cast<int64_t>(a.words) * n + e] = make_double2(xr, xi);
  }
  for (int off = 32; off > 0; off >>= 1) errors += __shfl_down(errors, off, 64);
  if ((tid & 63) == 0) atomicAdd(red, errors);
  __syncthreads();
  if (tid == 0) a.errors[local_drop] = red[0];
}

}  // namespace

extern "C" int hpx_run_batch_f64(const hpx_link* link_host, const int32_t* delays, const double* path_gains,
                                 uint64_t seed, int64_t first_drop, int64_t num_drops, const double* noise_power,
                                 int32_t* errors, hpx_c128* equalized, void* stream) {
  HPX_REQUIRE(link_host && delays && path_gains && noise_power && errors, "hpx_run_batch_f64: null pointer");
  HPX_REQUIRE(num_drops >= 0 && num_drops <= 0x7fffffff && first_drop >= 0 &&
                  first_drop + num_drops <= (int64_t(1) << 32),
              "hpx_run_batch_f64: invalid drop range");
  if (link_host->num_tx != 1 || link_host->num_rx != 1) {
    set_error("hpx_run_batch_f64: single-antenna links only (got %dx%d)", link_host->num_rx, link_host->num_tx);
    return HPX_ERR_UNSUPPORTED;
  }
  if (link_host->num_subcarriers > kF64MaxSubcarriers) {
    set_error("hpx_run_batch_f64: at most %d subcarriers (got %d)", kF64MaxSubcarriers, link_host->num_subcarriers);
    return HPX_ERR_UNSUPPORTED;
  }
  Plan plan;
  const int st = make_plan(link_host, nullptr, &plan, false, true);
  if (st != HPX_OK) return st;
  if (num_drops == 0) return HPX_OK;
  BatchArgs& a = plan.args;
  a.delays = delays;
  a.path_gains = path_gains;
  a.noise_power = noise_power;
  a.errors = errors;
  a.seed = seed;
  a.first_drop = first_drop;
  F64Layout g{};
  g.dx = a.maxd;
  g.frame = a.words * (a.n + a.cp);
  g.bits_words = static_cast<int>((static_cast<int64_t>(a.words) * a.n * a.bps + 31) / 32) + 1;
  // a round's rows of the tables; a frame too short for the tables of all sinusoids gets room for them (in groups
  // they cost two barriers each: 32 subcarriers, one word, 15 paths 177 us in groups of two, 119 at once)
  const int round = std::min(g.frame, kF64Round);
  const int row = (round + kF64Block - 1) / kF64Block + 2 * kF64Run;
  auto layout = [&](int work) {
    int64_t o = 0;
    auto take = [&](int64_t bytes) {
      const int at = static_cast<int>(o);
      o += align16(bytes);
      return at;
    };
    // the prologue's uniforms alias the transmit buffer where it is long enough, which it is for every
    // frame but the shortest; the sinusoids' tables alias the receive buffer
    const int64_t uni_elems = (static_cast<int64_t>(a.nnorm) + 1) / 2;  // in complex128 values
    g.work = work;
    g.off_sos = take(static_cast<int64_t>(a.paths) * a.terms * 3 * sizeof(double));
    g.off_tw = take(static_cast<int64_t>(a.n) * sizeof(double2));
    g.off_x = take(std::max<int64_t>(g.dx + g.frame, uni_elems) * sizeof(double2));
    g.off_y = take(static_cast<int64_t>(work) * sizeof(double2));
    g.off_abar = take(static_cast<int64_t>(a.paths) * a.words * sizeof(double2));
    g.off_bits = take(static_cast<int64_t>(g.bits_words) * sizeof(uint32_t));
    g.off_red = take(16);
    // (a frame has at least 32 samples: one term's table always fits)
    g.term_group = std::max(1, std::max(round, std::min(work, kF64Round)) / row);
    g.bytes = o;
  };
  layout(std::max(g.frame, std::min(a.terms * row, kF64Tables)));
  if (g.bytes > kMaxLds) layout(g.frame);
  if (g.bytes > kMaxLds) {
    set_error("hpx_run_batch_f64: %lld bytes of LDS per drop exceed a CU's %lld", static_cast<long long>(g.bytes),
              static_cast<long long>(kMaxLds));
    return HPX_ERR_UNSUPPORTED;
  }
  const auto kernel = g.frame <= kF64Threads ? f64_drop_kernel<1> : f64_drop_kernel<kF64Run>;
  if (!ensure_lds(reinterpret_cast<const void*>(kernel), g.bytes)) {
    set_error("hpx_run_batch_f64: %lld bytes of LDS per workgroup not available", static_cast<long long>(g.bytes));
    return HPX_ERR_UNSUPPORTED;
  }
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(num_drops)), dim3(kF64Threads),
                     static_cast<size_t>(g.bytes), static_cast<hipStream_t>(stream), a,
                     g, reinterpret_cast<double2*>(equalized));
  return check_launch("hpx_run_batch_f64");
}

