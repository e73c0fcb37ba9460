// liblensim: HIP kernels for gfx950 and the C ABI declared in include/lensim.h.
//
// Pipeline of one batched image / likelihood call (all on one stream):
//   prep_psf_kernel  kwargs slots -> per-(image, profile) records (+ EPL series
//                    coefficients), float64 and float32 copies; in the same
//                    launch the PSF preparation: the flipped kernel for the
//                    direct convolution, or the fp16 hi/lo B fragments of the
//                    matrix-core convolution
//   render_kernel /  one thread per pixel: s x s sub-rays generated from the
//   render_fast_...  grid description, ray shooting through every deflector,
//                    source light at the deflected position and lens light at
//                    the ray, mean over the sub-pixel block, x pixel_width^2 x
//                    flux_scaling (the fast kernel for compile-time profile
//                    lists of the common model family)
//   conv_kernel /    'same' convolution (zero or edge padding): LDS-tiled
//   conv_mfma_kernel direct stencil in the compute type, or fp16 hi/lo split
//                    products on the matrix cores (mixed form); optionally
//                    fused with the per-pixel chi^2 and a block reduction
//   logl_kernel      fixed-order sum of the per-tile chi^2 partials
#include <hip/hip_runtime.h>

#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <mutex>
#include <type_traits>

#include "grad.hpp"
#include "profiles.hpp"

using namespace lensim;

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int hip_fail(hipError_t e, const char *where) {
  return fail(LENSIM_EDEVICE, "%s: %s", where, hipGetErrorString(e));
}

inline size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

// ---- bounds-checked build (-DLENSIM_BOUNDS_CHECK, liblensim_checked.so) ----
// Each entry point registers the buffers of its call (workspace, parameters,
// data, PSF, outputs) before its launches.  A checked access AT(p, i) tests
// that element i of p lies inside one of them; one that does not is diverted
// to a private sink and the first such access's source line is recorded, so
// the kernel touches no memory outside the call's buffers and still ends
// normally.  After the call the entry point waits for its stream and returns
// LENSIM_EDEVICE naming that line, and clears the ranges again: a call that
// registers none (graph capture, which cannot wait for its stream) runs
// unchecked.  In the normal build AT(p, i) is p[i].
constexpr int kMaxRanges = 24;
struct CheckRanges {
  int n;
  unsigned long long lo[kMaxRanges], hi[kMaxRanges];
};
#ifdef LENSIM_BOUNDS_CHECK
__constant__ CheckRanges g_ranges;
__device__ unsigned int g_violation;
__device__ __align__(16) unsigned char g_sink[64];

__device__ __forceinline__ bool in_ranges(const void *p, size_t n) {
  const unsigned long long a = reinterpret_cast<unsigned long long>(p);
  if (g_ranges.n == 0) return true;  // no ranges registered: unchecked
  for (int r = 0; r < g_ranges.n; ++r)
    if (a >= g_ranges.lo[r] && a + n <= g_ranges.hi[r]) return true;
  return false;
}

__device__ __noinline__ void report_violation(int line) { atomicCAS(&g_violation, 0u, unsigned(line)); }

template <typename T>
__device__ __forceinline__ T &checked_at(T *p, size_t i, int line) {
  if (!in_ranges(p + i, sizeof(T))) {
    report_violation(line);
    return *reinterpret_cast<T *>(g_sink);
  }
  return p[i];
}
#define AT(p, i) checked_at((p), size_t(i), __LINE__)
// a base pointer and extent the kernel reads from with fixed offsets (records)
#define CHECK_SPAN(p, n) \
  do {                   \
    if (!in_ranges((p), (n))) report_violation(__LINE__); \
  } while (0)
#else
#define AT(p, i) (p)[i]
#define CHECK_SPAN(p, n) \
  do {                   \
  } while (0)
#endif

// while a call is captured into a graph (lensim_graph_capture_loglike) no
// timing events are recorded (they would become nodes of the graph) and the
// checked build registers no ranges (it would have to wait for the stream)
thread_local bool g_capturing = false;

// The buffers of one call, for the checked build (no-ops otherwise).
class CallRanges {
 public:
  void add(const void *p, size_t bytes) {
    if (!p || !bytes) return;
    if (r_.n >= kMaxRanges) {
      overflow_ = true;
      return;
    }
    r_.lo[r_.n] = reinterpret_cast<unsigned long long>(p);
    r_.hi[r_.n] = r_.lo[r_.n] + bytes;
    ++r_.n;
  }
#ifdef LENSIM_BOUNDS_CHECK
  int begin(hipStream_t st) {
    if (g_capturing) return LENSIM_OK;
    if (overflow_) return fail(LENSIM_EINVAL, "bounds check: more than %d buffers in one call", kMaxRanges);
    const unsigned int zero = 0;
    hipError_t e = hipMemcpyToSymbolAsync(HIP_SYMBOL(g_ranges), &r_, sizeof(r_), 0, hipMemcpyHostToDevice, st);
    if (e == hipSuccess)
      e = hipMemcpyToSymbolAsync(HIP_SYMBOL(g_violation), &zero, sizeof(zero), 0, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);  // the host copies above read r_ and zero
    return e == hipSuccess ? LENSIM_OK : hip_fail(e, "bounds check set-up");
  }
  int end(hipStream_t st, int rc) {
    if (g_capturing) return rc;
    unsigned int line = 0;
    const int none = 0;
    hipError_t e = hipStreamSynchronize(st);
    if (e == hipSuccess) e = hipMemcpyFromSymbol(&line, HIP_SYMBOL(g_violation), sizeof(line));
    if (e == hipSuccess) e = hipMemcpyToSymbol(HIP_SYMBOL(g_ranges), &none, sizeof(none));
    if (rc) return rc;
    if (e != hipSuccess) return hip_fail(e, "bounds check");
    if (line)
      return fail(LENSIM_EDEVICE, "bounds check: an access at lensim.hip:%u fell outside the call's buffers", line);
    return LENSIM_OK;
  }
#else
  int begin(hipStream_t) { return LENSIM_OK; }
  int end(hipStream_t, int rc) { return rc; }
#endif

 private:
  CheckRanges r_{};
  bool overflow_ = false;
};

constexpr int kWin = 8;  // register window (outputs per thread) of the convolution
constexpr int kGradPix = 4;  // pixels per thread of the gradient kernel
constexpr size_t kMaxLds = 160 * 1024;  // LDS per workgroup on gfx950

// ---- optional kernel timing (lensim_timing_*) ----
struct TimedCall {
  hipEvent_t ev[3];  // before render, after render / before conv, after conv
};
bool g_timing = false;
TimedCall *g_calls = nullptr;
int g_ncalls = 0, g_capcalls = 0;

hipEvent_t timing_event(int slot) {
  if (!g_timing) return nullptr;
  if (slot == 0) {
    if (g_ncalls == g_capcalls) {
      const int cap = g_capcalls ? 2 * g_capcalls : 256;
      TimedCall *n = static_cast<TimedCall *>(realloc(g_calls, sizeof(TimedCall) * cap));
      if (!n) return nullptr;
      for (int i = g_capcalls; i < cap; ++i)
        for (int k = 0; k < 3; ++k) n[i].ev[k] = nullptr;
      g_calls = n;
      g_capcalls = cap;
    }
    ++g_ncalls;
  }
  TimedCall &c = g_calls[g_ncalls - 1];
  if (!c.ev[slot] && hipEventCreate(&c.ev[slot]) != hipSuccess) c.ev[slot] = nullptr;
  return c.ev[slot];
}


void timing_mark(int slot, hipStream_t st) {
  if (!g_timing || g_capturing) return;
  hipEvent_t e = timing_event(slot);
  if (e) (void)hipEventRecord(e, st);
}

// Record index space: [0, n_lens) inline deflectors, [n_lens, n_defl) bulk
// deflectors, [n_defl, n_defl + n_source) source light, then lens light.
// types[] holds the inline lens, source and lens-light types (no bulk).
struct ModelArgs {
  int32_t n_lens, n_bulk, n_defl, n_source, n_light, n_prof, n_epl, has_halo, bulk_type;
  int32_t has_nie_nfw;  // an SIE / NIE or NFW deflector (inline or bulk), or halos on several planes: the float
                        // form deflects SIE / NIE and the NFW family in double
  SubSteps sub;         // sub-ray steps of the call's grid, for the records (with_grid); zero without a grid
  int32_t unit_amp;     // the light profiles' records take amp = 1 (the linear solve's responses)
  const int32_t *bulk_types;
  int32_t types[LENSIM_MAX_PROFILES];
  int32_t epl_index[LENSIM_MAX_PROFILES];
  double alpha_scaling, flux_scaling;
  // multi-plane ray tracing (mp_n == 0: single plane)
  int32_t mp_n;
  const int32_t *mp_order;
  const double *mp_tij, *mp_tz, *mp_r2p;
  int64_t mp_stride;
  int32_t mp_runs;      // the caller's bound on the plane runs (max_runs), else the deflectors
};

__host__ __device__ inline int type_of(const ModelArgs &m, int k) {
  if (k < m.n_lens) return m.types[k];
  if (k < m.n_defl) return m.bulk_type ? m.bulk_type : m.bulk_types[k - m.n_lens];
  return m.types[k - m.n_bulk];
}

struct Layout {
  size_t recd, recf, coefd, coeff, dcoefd, dcoeff, psf, lowres, partial, blkmax, bfrag;
  size_t gmodel, glow, gpart;  // gradient: dlogL/dmodel, dlogL/dlowres, per-block partial gradients
  size_t gbeta;                // gradient: dS/dbeta of the sources at every ray (0: none)
  size_t beta;                 // gradient of a bulk or multi-plane list: beta at every ray (0: none)
  size_t gpart_mp, gstate;     // ... its deflectors' partial sums and the rays' adjoints (0: none)
  size_t gpad, gext;           // edge-padded PSF adjoint: padded dlogL/dmodel and its correlation
  size_t gchr, glu;            // supersampled convolution adjoint buffers
  size_t mp_tab;               // several planes: the plane runs (mp_runs_kernel)
  size_t hr, chr, lowu, lowc, psf_low;  // supersampled convolution: ray fluxes, their convolution,
                                        // pooled unconvolved image and its low-resolution convolution
  size_t total;
  int n_tiles;
};

// Convolution tile shape (outputs per block): TX columns, TY rows; each
// thread owns kWin consecutive rows of one column, so a block has
// TX * TY / kWin threads and lanes of a wave read consecutive LDS words.
template <typename T>
struct ConvTile {
  static constexpr int TY = 32, TX = 32;  // 128 threads
};

// kernel height padded to a multiple of the register window
int kyp_of(int ky) { return (ky + kWin - 1) / kWin * kWin; }

// ---- MFMA convolution geometry (mixed form) ----
// Each kernel row a contributes D(16x16) += A(16x32k) B(32k x16) per output
// tile, with A = 16 image rows of the padded tile and B[k][n] = Kf[a][k - n]
// (the band of kernel row a).  nks K-steps of 32 cover 16 + kx - 1 columns.
constexpr int kMfWaves = 4;  // waves per block, each 16 output rows
constexpr int kMfTY = 16 * kMfWaves;
// 16-column tiles per wave: TL in [2, 4], chosen per call (mfma_plan)
int mfma_nks(int kx) { return (16 + kx - 1 + 31) / 32; }
constexpr int kMfMaxNks = 4;  // kernels up to 113 columns
// Kernel rows per unrolled loop body (and per float -> double fold): the B
// fragments of that many rows (about 4 K-steps) are in flight at once.
constexpr int mfma_unroll(int nks) { return (4 + nks - 1) / nks; }
// B-fragment steps: ky padded to a multiple of the unroll with zero rows.
int mfma_steps(int kx, int ky) {
  const int nks = mfma_nks(kx), u = mfma_unroll(nks);
  return (ky + u - 1) / u * u * nks;
}
int mfma_tw(int kx, int tl) { return 16 * (tl - 1) + 32 * mfma_nks(kx); }
// LDS row stride in halves.  The A reads (ds_read_b128, lane l at row l % 16,
// 16-byte column l / 16) are free of bank conflicts when the stride in dwords
// is 8 (mod 16), as measured on gfx950 (strides of 4 or 12 (mod 16) dwords
// conflict, 0 (mod 64) serialises).  tw = 16 (tl - 1) + 32 nks halves: for
// even tl it is 16 (mod 32) and unpadded; for tl = 3 it is padded by 16.
int mfma_ls(int kx, int tl) {
  const int tw = mfma_tw(kx, tl);
  return tw % 32 == 16 ? tw : tw + 16;
}
size_t mfma_smem(int kx, int ky, int tl) {
  return size_t(kMfTY + ky - 1) * mfma_ls(kx, tl) * 2 * sizeof(_Float16);
}

// ---- convolution of the FP64 form ----
// conv_f64_kernel's LDS: rows of a tile (the register groups are read whole,
// past the rows in use), doubles of the tile (later the waves' sums), and
// with the weights in bytes.
int conv_f64_rows(int ky, int r, int h) {
  const int used = 2 * r * h + ky - 1, read = (2 * h - 1) * r + 24 + ky / 8 * 8;
  return used > read ? used : read;
}
__host__ __device__ inline int conv_f64_tile(int kx, int th, int r, int h, int cls) {
  const int t = th * (32 + kx - 1) + 1, sums = 64 * cls * h * r;
  return (t > sums ? t : sums) & ~1;
}
size_t conv_f64_smem(int kx, int ky, int r, int h, int cls, bool gw) {
  return (size_t(conv_f64_tile(kx, conv_f64_rows(ky, r, h), r, h, cls)) + (gw ? 0 : size_t(kx) * kyp_of(ky))) *
         sizeof(double);
}

// Blocks of 64 rows x 16 tl columns.  All of a call's blocks are resident at
// once on this workload's sizes, so the time is that of the busiest CU:
// ceil(blocks / CUs) blocks of tl wave-tiles.  tl is the one in [2, 4] with
// the least such load (ties to the wider tile, which re-reads fewer A
// fragments): for 180^2 x 64 images, 768 blocks of 48 columns (3 per CU)
// against 576 of 64 (2.25 per CU, so 3 on some).
struct MfmaPlan {
  int tl, n_tiles_x, n_tiles;
};
int cu_count() {
  static int n = 0;
  if (n == 0) {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
      n = v;
    else
      n = 256;
  }
  return n;
}
MfmaPlan mfma_plan(int nx, int ny, int n_img, int kx, int ky) {
  MfmaPlan best{0, 0, 0};
  long best_load = 0;
  const int cus = cu_count();
  for (int tl = 4; tl >= 2; --tl) {
    if (mfma_smem(kx, ky, tl) > kMaxLds) continue;
    const int ntx = (nx + 16 * tl - 1) / (16 * tl), nt = ntx * ((ny + kMfTY - 1) / kMfTY);
    const long blocks = long(nt) * n_img;
    const long load = (blocks + cus - 1) / cus * tl;
    if (best.tl == 0 || load < best_load) {
      best = MfmaPlan{tl, ntx, nt};
      best_load = load;
    }
  }
  return best;
}

// 16 x 16 output tiles of an image (the matrix-core convolution's chi^2 partials)
int n16_tiles(int nx, int ny) { return ((nx + 15) / 16) * ((ny + 15) / 16); }

template <typename T>
int n_tiles_of(int nx, int ny) {
  const int tx = (nx + ConvTile<T>::TX - 1) / ConvTile<T>::TX;
  const int ty = (ny + ConvTile<T>::TY - 1) / ConvTile<T>::TY;
  return tx * ty;
}

// Supersampled convolution plan (lensim_psf.supersampled on a grid with s > 1).
struct SSPlan {
  int on = 0;        // convolve on the supersampled grid
  int s = 1;
  int kxl = 0, kyl = 0;  // low-resolution split kernel (0: none)
};

// The plane runs of a multi-plane model (mp_runs_kernel), int32 per set of
// plane arrays (one for the batch when they are shared): [0] the number of
// runs n, [1] whether a deflector is on several planes, [2] whether the bulk
// list holds subhalos and linear deflectors only, then run starts
// [n + 1 <= mp_n], the run of each plane [mp_n - 1], the plane of each
// deflector [n_defl], and the deflector of each plane with its type
// [mp_n - 1] (index + 2^24 type).
__host__ __device__ inline int mp_tab_ints(const ModelArgs &m) { return 1 + 3 * m.mp_n + m.n_defl; }
size_t mp_tab_sets(const ModelArgs &m, int n_img) { return m.mp_stride ? size_t(n_img) : 1; }

Layout layout(const ModelArgs &m, int nx, int ny, int kx, int ky, int n_img, int precision,
              const SSPlan &ss = SSPlan()) {
  Layout L{};
  const size_t tsz = precision == LENSIM_MIXED ? 4 : 8;
  size_t off = 0;
  const size_t nrec = size_t(n_img) * m.n_prof * kRec;
  L.recd = off;
  off = align256(off + nrec * 8);
  L.recf = off;
  off = align256(off + nrec * 4);
  const size_t ncoef = size_t(n_img) * m.n_epl * LENSIM_EPL_NMAX;
  L.coefd = off;
  off = align256(off + ncoef * 8);
  L.coeff = off;
  off = align256(off + ncoef * 4);
  L.dcoefd = off;
  off = align256(off + ncoef * 8);
  L.dcoeff = off;
  off = align256(off + ncoef * 4);
  L.psf = off;
  off = align256(off + size_t(kx) * kyp_of(ky) * 8);
  L.lowres = off;
  off = align256(off + size_t(n_img) * nx * ny * tsz);
  L.n_tiles = precision == LENSIM_MIXED ? n_tiles_of<float>(nx, ny) : n_tiles_of<double>(nx, ny);
  const size_t npix = size_t(nx) * ny, npix_r = ss.on ? npix * ss.s * ss.s : npix;  // rendered pixels
  L.partial = off;  // per-tile (or per-block, or per 16 x 16 tile) chi^2 partials
  {
    size_t np_ = L.n_tiles;
    np_ = np_ > (npix + 255) / 256 ? np_ : (npix + 255) / 256;
    np_ = np_ > size_t(n16_tiles(nx, ny)) ? np_ : size_t(n16_tiles(nx, ny));
    off = align256(off + size_t(n_img) * np_ * 8);
  }
  L.blkmax = off;  // per render block max |value|, [n_img][ceil(rendered pixels / 256)]
  off = align256(off + size_t(n_img) * ((npix_r + 255) / 256) * 4);
  L.hr = L.chr = L.lowu = L.lowc = L.psf_low = off;
  if (ss.on) {
    L.hr = off;
    off = align256(off + size_t(n_img) * npix_r * tsz);
    L.chr = off;
    off = align256(off + size_t(n_img) * npix_r * tsz);
    if (ss.kxl > 0) {
      L.lowu = off;
      off = align256(off + size_t(n_img) * npix * tsz);
      L.lowc = off;
      off = align256(off + size_t(n_img) * npix * tsz);
      L.psf_low = off;
      off = align256(off + size_t(ss.kxl) * kyp_of(ss.kyl) * 8);
    }
  }
  L.mp_tab = off;
  if (m.mp_n > 0) off = align256(off + mp_tab_sets(m, n_img) * size_t(mp_tab_ints(m)) * 4);
  L.bfrag = off;  // int exponent (16 B slot) then the MFMA B fragments
  if (precision == LENSIM_MIXED) off = align256(off + 16 + size_t(mfma_steps(kx, ky)) * 2 * 64 * 16);
  L.total = off;
  return L;
}

// Work plan of the gradient of a bulk or multi-plane deflector list over
// `rays` rays an image (adjoint kernels, then defl_grad_kernel).  The adjoint
// kernels keep four doubles per ray and run: per_img of them an image, at most
// kStoreMost (1 GiB) together: `imgs` images at a time, and an image that takes
// more by itself in `rounds` of its rays.  `runs` is the caller's bound on a
// multi-plane model's runs (lensim_multiplane.max_runs), without one a run per
// plane: the kernels take as many rays a round as the runs there are allow, and
// what the plan has too many of ends at once.  splits: pieces a deflector's rays
// of a round are cut into (a partial sum each, to which the rounds add): so that
// about 2048 waves, and up to 16384 of 2048 rays, share an image's deflectors,
// each 512 rays or, of up to 128 splits, 64 (two deflectors and 60^2 rays 85 us a
// call with 512, 67 with 64; 100^2 x 4 108, 102 and, of 625 splits, 113).  Nothing but `imgs` depends on the batch, so a list's sums
// on one plane have the same order in any.  The partial sums take imgs n splits
// 64 B: with a pair of deflectors a wave at most 2 MB an image beside one sum
// for each deflector.
constexpr size_t kStoreMost = size_t(1) << 25;
struct DeflGradPlan {
  size_t per_img;
  int imgs, rounds, splits, n, runs;  // n: deflectors (planes, or the bulk list)
};
DeflGradPlan defl_grad_plan(const ModelArgs &m, size_t rays, int n_img) {
  DeflGradPlan p{0, n_img, 1, 1, m.mp_n ? m.mp_n - 1 : m.n_bulk, 1};
  if (p.n == 0) return p;
  if (m.mp_n) p.runs = m.mp_runs;
  const size_t all = (rays + 63) / 64 * 64 * p.runs;
  p.per_img = all < kStoreMost ? all : kStoreMost;
  const size_t cap = p.per_img / p.runs / 64 * 64, fit = kStoreMost / p.per_img;
  p.rounds = int((rays + cap - 1) / cap);
  if (fit < size_t(n_img)) p.imgs = int(fit);
  const size_t pairs = size_t(p.n + 1) / 2;
  auto over = [](size_t a, size_t b) { return (a + b - 1) / b; };
  size_t sp = over(rays, 2048);
  if (sp > over(16384, pairs)) sp = over(16384, pairs);
  if (sp < over(2048, pairs)) sp = over(2048, pairs);
  const size_t most = over(rays, 512) > 128 ? over(rays, 512) : over(rays, 64) < 128 ? over(rays, 64) : 128;
  if (sp > most) sp = most;
  p.splits = int(sp < 2048 ? sp : 2048);
  return p;
}

// Layout of lensim_loglike_grad: the image layout plus the gradient buffers
// (on the ray grid when the convolution is supersampled).
Layout grad_layout(const ModelArgs &m, int nx, int ny, int kx, int ky, int n_img, int precision, int edge,
                   const SSPlan &ss, int s) {
  Layout L = layout(m, nx, ny, kx, ky, n_img, precision, ss);
  const size_t tsz = precision == LENSIM_MIXED ? 4 : 8;
  const size_t npix = size_t(nx) * ny;
  const int cs = ss.on ? ss.s : 1;
  const size_t npix_r = npix * cs * cs;  // pixels of the grid the convolution runs on
  size_t off = L.total;
  L.gmodel = off;
  off = align256(off + size_t(n_img) * npix * tsz);
  L.glow = off;
  off = align256(off + size_t(n_img) * npix_r * tsz);
  L.gpart = off;
  off = align256(off + size_t(n_img) * m.n_prof * ((npix_r + 256 * kGradPix - 1) / (256 * kGradPix)) *
                           LENSIM_NPARAM * 8);
  L.gbeta = L.beta = L.gpart_mp = L.gstate = 0;
  const size_t rays = npix_r * (ss.on ? 1 : size_t(s) * s);
  const bool list = m.mp_n > 0 || m.n_bulk > 0;
  if (m.n_lens > 0 && m.mp_n == 0 && m.n_source > 0) {
    L.gbeta = off;
    off = align256(off + size_t(n_img) * rays * 2 * tsz);
  }
  if (list && m.n_source > 0) {
    L.beta = off;
    off = align256(off + size_t(n_img) * rays * 2 * tsz);
  }
  if (list && m.n_defl > 0) {
    const DeflGradPlan p = defl_grad_plan(m, rays, n_img);
    L.gpart_mp = off;
    off = align256(off + size_t(p.imgs) * p.n * p.splits * LENSIM_NPARAM * 8);
    L.gstate = off;
    off = align256(off + size_t(p.imgs) * p.per_img * 32);
  }
  L.gpad = L.gext = L.gchr = L.glu = off;
  if (edge) {  // extended domain (ny cs + ky - 1) x (nx cs + kx - 1)
    const size_t next = size_t(nx * cs + kx - 1) * (ny * cs + ky - 1);
    L.gpad = off;
    off = align256(off + size_t(n_img) * next * tsz);
    L.gext = off;
    off = align256(off + size_t(n_img) * next * tsz);
  }
  if (ss.on) {
    L.gchr = off;  // dlogL / d(convolved rays)
    off = align256(off + size_t(n_img) * npix_r * tsz);
    L.glu = off;   // dlogL / d(pooled unconvolved rays), split kernel
    off = align256(off + size_t(n_img) * npix * tsz);
  }
  L.total = off;
  return L;
}

bool bulk_type_ok(int t) {
  return t == LENSIM_NULL || t == LENSIM_SIE || t == LENSIM_NIE || t == LENSIM_NFW || t == LENSIM_TNFW ||
         t == LENSIM_SHEAR || t == LENSIM_CONVERGENCE;
}

int model_args(const lensim_model *model, ModelArgs &m) {
  if (!model) return fail(LENSIM_EINVAL, "model is NULL");
  m = ModelArgs{};
  m.n_lens = model->n_lens;
  m.n_source = model->n_source;
  m.n_light = model->n_lens_light;
  m.n_bulk = model->n_bulk;
  if (m.n_lens < 0 || m.n_source < 0 || m.n_light < 0 || m.n_bulk < 0)
    return fail(LENSIM_EINVAL, "negative profile count");
  const int n_inline = m.n_lens + m.n_source + m.n_light;
  if (n_inline > LENSIM_MAX_PROFILES)
    return fail(LENSIM_EINVAL, "%d profiles exceed LENSIM_MAX_PROFILES=%d", n_inline, LENSIM_MAX_PROFILES);
  if (m.n_bulk > (1 << 20)) return fail(LENSIM_EINVAL, "n_bulk %d too large", m.n_bulk);
  m.n_defl = m.n_lens + m.n_bulk;
  m.n_prof = n_inline + m.n_bulk;
  for (int k = 0; k < n_inline; ++k) {
    const int t = model->types[k];
    m.types[k] = t;
    m.epl_index[k] = -1;
    const bool lens = k < m.n_lens;
    const bool lens_ok = t == LENSIM_EPL || t == LENSIM_SIE || t == LENSIM_NIE || t == LENSIM_NFW ||
                         t == LENSIM_TNFW || t == LENSIM_SHEAR || t == LENSIM_CONVERGENCE;
    const bool light_ok = t == LENSIM_SERSIC || t == LENSIM_SERSIC_ELLIPSE || t == LENSIM_GAUSSIAN;
    if (lens && !lens_ok) return fail(LENSIM_EUNSUPPORTED, "profile %d: type %d is not a supported deflector", k, t);
    if (!lens && !light_ok)
      return fail(LENSIM_EUNSUPPORTED, "profile %d: type %d is not a supported light profile", k, t);
    if (t == LENSIM_EPL) m.epl_index[k] = m.n_epl++;
    if (t == LENSIM_NFW || t == LENSIM_TNFW) m.has_halo = 1;
    if (lens && (t == LENSIM_SIE || t == LENSIM_NIE || t == LENSIM_NFW)) m.has_nie_nfw = 1;
  }
  if (m.n_bulk > 0) {
    m.bulk_type = model->bulk_type;
    m.bulk_types = model->d_bulk_types;
    if (!bulk_type_ok(m.bulk_type))
      return fail(LENSIM_EUNSUPPORTED, "bulk deflector type %d not supported (SIE, NIE, NFW, TNFW, SHEAR, CONVERGENCE)",
                  m.bulk_type);
    if (m.bulk_type == LENSIM_NULL && !m.bulk_types)
      return fail(LENSIM_EINVAL, "mixed bulk deflectors need d_bulk_types");
    if (m.bulk_type == LENSIM_NFW || m.bulk_type == LENSIM_TNFW || m.bulk_type == LENSIM_NULL) m.has_halo = 1;
    if (m.bulk_type == LENSIM_SIE || m.bulk_type == LENSIM_NIE || m.bulk_type == LENSIM_NFW ||
        m.bulk_type == LENSIM_NULL)
      m.has_nie_nfw = 1;
  }
  m.alpha_scaling = model->alpha_scaling;
  m.flux_scaling = model->flux_scaling;
  if (const lensim_multiplane *mp = model->multiplane) {
    if (mp->n_planes != m.n_defl + 1)
      return fail(LENSIM_EINVAL, "multiplane.n_planes %d must be the %d deflectors + 1", mp->n_planes, m.n_defl);
    if ((m.n_defl > 0 && !mp->d_order) || !mp->d_T_ij || !mp->d_T_z || !mp->d_r2p)
      return fail(LENSIM_EINVAL, "multiplane arrays are NULL");
    if (mp->stride != 0 && mp->stride < mp->n_planes) return fail(LENSIM_EINVAL, "multiplane stride too small");
    m.mp_n = mp->n_planes;
    m.mp_order = mp->d_order;
    m.mp_tij = mp->d_T_ij;
    m.mp_tz = mp->d_T_z;
    m.mp_r2p = mp->d_r2p;
    m.mp_stride = mp->stride;
    m.mp_runs = mp->max_runs > 0 && mp->max_runs < m.n_defl ? mp->max_runs : m.n_defl;
    // with several planes a deflector's error moves the rays at every later
    // plane, where a strong lens magnifies it: the float form's render and
    // gradient kernels deflect the NFW family in double there too (the float
    // TNFW left logL 2e-6 off)
    if (m.has_halo) m.has_nie_nfw = 1;
  }
  return LENSIM_OK;
}

// ------------------------------------------------------------- kernels ---

__device__ inline bool bulk_type_ok_dev(int t) {
  return t == LENSIM_NULL || t == LENSIM_SIE || t == LENSIM_NIE || t == LENSIM_NFW || t == LENSIM_TNFW ||
         t == LENSIM_SHEAR || t == LENSIM_CONVERGENCE;
}

// Record (and EPL coefficients) number idx < n_img * n_prof, profile-major
// (idx = k * n_img + img), so the lanes of a wave share one profile type and
// take one branch of prepare_record; records are stored [img][k].
__device__ void prep_one(const ModelArgs &m, const double *__restrict__ params, int n_img, int idx,
                         double *__restrict__ recd, float *__restrict__ recf, double *__restrict__ coefd,
                         float *__restrict__ coeff, double *__restrict__ dcoefd, float *__restrict__ dcoeff) {
  const int k = idx / n_img, img = idx - k * n_img;
  const int ri = img * m.n_prof + k;
  if (k >= m.n_lens && k < m.n_defl && !m.bulk_type) CHECK_SPAN(m.bulk_types + (k - m.n_lens), sizeof(int32_t));
  int type = type_of(m, k);
  if (k >= m.n_lens && k < m.n_defl && !bulk_type_ok_dev(type)) type = LENSIM_NULL;
  const double *p = params + size_t(ri) * LENSIM_NPARAM;
  CHECK_SPAN(p, LENSIM_NPARAM * sizeof(double));
  double rec[kRec];
  double *coef = nullptr, *dcoef = nullptr;
  float *cf = nullptr, *dcf = nullptr;
  const int e = k < m.n_lens ? m.epl_index[k] : -1;
  if (e >= 0) {
    const size_t co = (size_t(img) * m.n_epl + e) * LENSIM_EPL_NMAX;
    coef = coefd + co;
    cf = coeff + co;
    CHECK_SPAN(coef, LENSIM_EPL_NMAX * sizeof(double));
    CHECK_SPAN(cf, LENSIM_EPL_NMAX * sizeof(float));
    if (dcoefd) {
      dcoef = dcoefd + co;
      dcf = dcoeff + co;
      CHECK_SPAN(dcoef, LENSIM_EPL_NMAX * sizeof(double));
      CHECK_SPAN(dcf, LENSIM_EPL_NMAX * sizeof(float));
    }
  }
  double q[LENSIM_NPARAM];
#pragma unroll
  for (int i = 0; i < LENSIM_NPARAM; ++i) q[i] = (i == 0 && m.unit_amp && k >= m.n_defl) ? 1.0 : p[i];
  prepare_record(type, q, rec, coef, m.sub, dcoef, cf, dcf);
  for (int i = 0; i < kRec; ++i) {
    AT(recd, size_t(ri) * kRec + i) = rec[i];
    AT(recf, size_t(ri) * kRec + i) = float(rec[i]);
  }
  if (type == LENSIM_EPL) {  // series lengths as int bits in the float copy
    AT(recf, size_t(ri) * kRec + EPL_NMAX) = __int_as_float(int(rec[EPL_NMAX]));
    AT(recf, size_t(ri) * kRec + EPL_NZ) = __int_as_float(int(rec[EPL_NZ]));
    AT(recf, size_t(ri) * kRec + EPL_NF) = __int_as_float(int(rec[EPL_NF]));
  }
}

__global__ void prep_kernel(ModelArgs m, const double *__restrict__ params, int n_img, double *__restrict__ recd,
                            float *__restrict__ recf, double *__restrict__ coefd, float *__restrict__ coeff,
                            double *__restrict__ dcoefd, float *__restrict__ dcoeff) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx < n_img * m.n_prof) prep_one(m, params, n_img, idx, recd, recf, coefd, coeff, dcoefd, dcoeff);
}

// Flip the kernel (so the convolution runs as a correlation) and store it
// transposed, column c of the flipped kernel contiguous: kt[c * kyp + a] =
// K[ky-1-a][kx-1-c], zero for a >= ky.
__device__ void psf_prep_one(const double *__restrict__ k, int kx, int ky, int kyp, double *__restrict__ out,
                             int flip, int idx) {
  const int c = idx / kyp, a = idx - c * kyp;
  if (!k) {  // identity kernel (no PSF / unconvolved)
    AT(out, idx) = (a == 0 && c == 0) ? 1.0 : 0.0;
    return;
  }
  // flip = 0 stores the kernel itself: the convolution then correlates with K,
  // which is the adjoint of convolving with K (zero padding)
  AT(out, idx) = (a < ky) ? (flip ? AT(k, (ky - 1 - a) * kx + (kx - 1 - c)) : AT(k, a * kx + c)) : 0.0;
}

__global__ void psf_prep_kernel(const double *__restrict__ k, int kx, int ky, int kyp, double *__restrict__ out,
                                int flip = 1) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx < kyp * kx) psf_prep_one(k, kx, ky, kyp, out, flip, idx);
}

template <typename T>
struct RecPtrs {
  const double *recd;
  const T *rect;
  const double *coefd;
  const T *coeft;
};

template <typename T>
__device__ __forceinline__ RecPtrs<T> rec_ptrs(const ModelArgs &m, const double *recd, const float *recf,
                                               const double *coefd, const float *coeff, int img) {
  RecPtrs<T> r;
  r.recd = recd + size_t(img) * m.n_prof * kRec;
  CHECK_SPAN(r.recd, size_t(m.n_prof) * kRec * sizeof(double));
  if constexpr (sizeof(T) == sizeof(float)) {
    r.rect = recf + size_t(img) * m.n_prof * kRec;
    CHECK_SPAN(r.rect, size_t(m.n_prof) * kRec * sizeof(float));
    r.coeft = coeff;
  } else {
    r.rect = r.recd;
    r.coeft = coefd;
  }
  r.coefd = coefd;
  return r;
}

// The deflection of the bulk list (records n_lens .. n_defl - 1) added to (ax, ay):
// every nw-th of them from the one `from`.
template <typename T, bool HALO, bool DBL = false, bool DBL_TNFW = DBL>
__device__ __forceinline__ void deflect_bulk(const ModelArgs &m, const RecPtrs<T> &rp, double x, double y,
                                             double &ax, double &ay, int from = 0, int nw = 1) {
  if (m.n_bulk == 0) return;
  if (m.bulk_type == LENSIM_TNFW) {
    // common case of substructure: one profile type, no per-deflector switch
    if constexpr (HALO) {
      for (int k = m.n_lens + from; k < m.n_defl; k += nw) {
        if constexpr (DBL_TNFW) tnfw_defl<double>(Rec<double>{rp.recd + k * kRec, rp.recd + k * kRec}, x, y, ax, ay);
        else tnfw_defl<T>(Rec<T>{rp.recd + k * kRec, rp.rect + k * kRec}, x, y, ax, ay);
      }
    }
    return;
  }
  for (int k = m.n_lens + from; k < m.n_defl; k += nw) {
    const int type = m.bulk_type ? m.bulk_type : AT(m.bulk_types, k - m.n_lens);
    const Rec<T> r{rp.recd + k * kRec, rp.rect + k * kRec};
    add_deflection<T, HALO, DBL, DBL_TNFW>(type == LENSIM_EPL ? LENSIM_NULL : type, r, nullptr, nullptr, x, y, ax, ay);
  }
}

template <typename T, bool HALO, bool DBL = false, bool DBL_TNFW = DBL>
__device__ __forceinline__ void deflect_all(const ModelArgs &m, const RecPtrs<T> &rp, int img, double x, double y,
                                            double &ax, double &ay) {
  for (int k = 0; k < m.n_lens; ++k) {
    const int type = m.types[k];
    const Rec<T> r{rp.recd + k * kRec, rp.rect + k * kRec};
    const int e = m.epl_index[k];
    const size_t co = (e >= 0) ? (size_t(img) * m.n_epl + e) * LENSIM_EPL_NMAX : 0;
    if (e >= 0) CHECK_SPAN(rp.coeft + co, LENSIM_EPL_NMAX * sizeof(T));
    add_deflection<T, HALO, DBL, DBL_TNFW>(type, r, rp.coefd + co, rp.coeft + co, x, y, ax, ay);
  }
  deflect_bulk<T, HALO, DBL, DBL_TNFW>(m, rp, x, y, ax, ay);
}

// One deflector k of type `type` (inline lens k < n_lens with its series coefficients, or bulk).
template <typename T, bool HALO, bool DBL, bool DBL_TNFW = DBL, bool SUB = false>
__device__ __forceinline__ void deflect_one(const ModelArgs &m, const RecPtrs<T> &rp, int img, int k, int type,
                                            double x, double y, double &ax, double &ay) {
  const Rec<T> r{rp.recd + k * kRec, rp.rect + k * kRec};
  size_t co = 0;
  if (!SUB && type == LENSIM_EPL) {
    co = (size_t(img) * m.n_epl + m.epl_index[k]) * LENSIM_EPL_NMAX;
    CHECK_SPAN(rp.coeft + co, LENSIM_EPL_NMAX * sizeof(T));
  }
  add_deflection<T, HALO, DBL, DBL_TNFW, SUB>(type, r, rp.coefd + co, rp.coeft + co, x, y, ax, ay);
}

// Source-plane position of the ray at angle (x, y) on a single plane:
// beta = theta - alpha_scaling * alpha.
template <typename T, bool HALO, bool DBL, bool DBL_TNFW = DBL>
__device__ __forceinline__ void trace_ray(const ModelArgs &m, const RecPtrs<T> &rp, int img, double x, double y,
                                          double &bx, double &by) {
  double ax = 0.0, ay = 0.0;
  deflect_all<T, HALO, DBL, DBL_TNFW>(m, rp, img, x, y, ax, ay);
  bx = x - ax * m.alpha_scaling;
  by = y - ay * m.alpha_scaling;
}

template <typename T>
__device__ __forceinline__ double light_sum(const ModelArgs &m, const RecPtrs<T> &rp, int k0, int k1, double x,
                                            double y) {
  double f = 0.0;
  for (int k = k0; k < k1; ++k) {
    const Rec<T> r{rp.recd + k * kRec, rp.rect + k * kRec};
    f += light_value<T>(m.types[k - m.n_bulk], r, x, y);
  }
  return f;
}

struct GridArgs {
  int nx, ny, s;
  double ra0, dec0, m00, m01, m10, m11;
  double scale;  // pixel_width^2 / s^2
  const uint8_t *mask;  // evaluation mask of the image pixels (NULL: all), [mask_ny][mask_nx]
  int mask_nx, mask_s;  // pixel (i, j) of this grid is mask pixel (i / mask_s, j / mask_s)
  // formed once on the host (grid_consts), so no thread divides: 1/s, the
  // first sub-ray's offset -1/2 + 1/(2 s) (make_subgrid, ImSim/Numerics/grid.py:60-62),
  // 1/nx and 1/s^2
  double inv_s, o0, inv_nx, inv_ss;
};

void grid_consts(GridArgs &g) {
  g.inv_s = 1.0 / g.s;
  g.o0 = -0.5 + 1.0 / (2.0 * g.s);
  g.inv_nx = 1.0 / g.nx;
  g.inv_ss = 1.0 / (double(g.s) * double(g.s));
}

// q = n / d and n - q d for 0 <= n < 2^30 and 1 <= d, from inv_d = 1/d in
// double: (n + 1/2) / d lies at least 1/(2d) from an integer, and the
// product's rounding error is below n 2^-52 < 2^-22 / d, so truncation gives q.
__device__ __forceinline__ int div_by(int n, int d, double inv_d, int &rem) {
  const int q = int((double(n) + 0.5) * inv_d);
  rem = n - q * d;
  return q;
}

// The same for n < 2^50.
__device__ __forceinline__ int64_t div_by64(int64_t n, int d, double inv_d, int &rem) {
  const int64_t q = int64_t((double(n) + 0.5) * inv_d);
  rem = int(n - q * d);
  return q;
}

// Whether grid pixel (i, j) is evaluated (RegularGrid flux_evaluate_indexes,
// ImSim/Numerics/grid.py:47-58: the rays of other pixels are not shot and
// their flux is zero).
__device__ __forceinline__ bool evaluated(const GridArgs &g, int i, int j) {
  return !g.mask || AT(g.mask, size_t(j / g.mask_s) * g.mask_nx + i / g.mask_s) != 0;
}

// The maximum over the 64 lanes of a wave (every lane active) of a
// non-negative float, by the integer max of the bit patterns (ordered as the
// values are): DPP quad permutations and row rotations give each row of 16
// lanes its maximum in every lane, readlane the four rows'.  Eight VALU
// instructions where a shuffle butterfly takes about fifty.
__device__ __forceinline__ float wave_max_nonneg(float x) {
  int v = __float_as_int(x);
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false));   // quad_perm [1, 0, 3, 2]
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false));   // quad_perm [2, 3, 0, 1]
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x124, 0xF, 0xF, false));  // row_ror:4
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x128, 0xF, 0xF, false));  // row_ror:8
  const int r = max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
                    max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
  return __int_as_float(r);
}

// The block's maximum of the threads' non-negative x (every thread of the
// block reaches this call) into *slot: one slot per block, no atomics.  The
// MFMA convolution scales its fp16 operands by the image maximum.
__device__ __forceinline__ void block_max_store(float x, float *slot) {
  __shared__ float wmax[256 / 64];
  const float mv = wave_max_nonneg(x);
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = mv;
  __syncthreads();
  if (threadIdx.x == 0) {
    float b = wmax[0];
    for (int w = 1; w < int(blockDim.x >> 6); ++w) b = fmaxf(b, wmax[w]);
    AT(slot, 0) = b;
  }
}

template <typename T, bool HALO, bool DBL>
__global__ __launch_bounds__(256) void render_kernel(ModelArgs m, GridArgs g, const double *__restrict__ recd,
                                                     const float *__restrict__ recf,
                                                     const double *__restrict__ coefd,
                                                     const float *__restrict__ coeff, unsigned flags,
                                                     T *__restrict__ out, float *__restrict__ blkmax) {
  const int img = blockIdx.y;
  const int npix = g.nx * g.ny;
  const int pix0 = blockIdx.x * blockDim.x + threadIdx.x;
  const bool active = pix0 < npix;
  const int pix = active ? pix0 : npix - 1;  // inactive lanes stay for the wave reduction
  int i;
  const int j = div_by(pix, g.nx, g.inv_nx, i);
  const RecPtrs<T> rp = rec_ptrs<T>(m, recd, recf, coefd, coeff, img);
  // pixel centre (lenstronomy grid_from_coordinate_transform order)
  const double ra_c = i * g.m00 + j * g.m01 + g.ra0;
  const double dec_c = i * g.m10 + j * g.m11 + g.dec0;
  const double inv_s = g.inv_s;
  const double o0 = g.o0;
  const bool do_src = (flags & LENSIM_IMAGE_SOURCE) && m.n_source > 0;
  const bool do_light = (flags & LENSIM_IMAGE_LENS_LIGHT) && m.n_light > 0;
  const int k_src0 = m.n_defl, k_src1 = m.n_defl + m.n_source, k_l1 = m.n_prof;
  double acc = 0.0;
  const bool eval = active && evaluated(g, i, j);
  for (int sy = 0; eval && sy < g.s; ++sy) {
    const double oy = o0 + sy * inv_s;
    for (int sx = 0; sx < g.s; ++sx) {
      const double ox = o0 + sx * inv_s;
      // make_subgrid offsets (ImSim/Numerics/grid.py:60-62)
      const double x = ra_c + g.m00 * ox + g.m01 * oy;
      const double y = dec_c + g.m10 * ox + g.m11 * oy;
      if (do_src) {
        double bx, by;
        trace_ray<T, HALO, DBL>(m, rp, img, x, y, bx, by);
        acc += light_sum<T>(m, rp, k_src0, k_src1, bx, by);
      }
      if (do_light) acc += light_sum<T>(m, rp, k_src1, k_l1, x, y);
    }
  }
  const T v = T(acc * (g.scale * m.flux_scaling));
  if (active) AT(out, size_t(img) * npix + pix) = v;
  if (blkmax) block_max_store(fabsf(float(v)), blkmax + size_t(img) * gridDim.x + blockIdx.x);
}

// The coordinates of a compile-time deflector that the sub-ray loop advances:
// Z = (q xr, yr) for the EPL, (xr, yr) for SIE / NIE (major-axis frame), the
// offset (dx, dy) from the centre for NFW.  They are affine in the ray
// position, so after their value at the pixel's first sub-ray each sub-ray
// adds a step (xs, ys) and each row a row step (xr_, yr_).
template <int TYPE>
struct DeflCoords {
  double a, b, sa, sb, ra, rb;
  __device__ __forceinline__ void init(const double *rd, const SubSteps &st, double x0, double y0) {
    const double dx = x0 - rd[R_CX], dy = y0 - rd[R_CY];
    if constexpr (TYPE == LENSIM_EPL) {
      const double c = rd[EPL_C], s = rd[EPL_S];
      a = rd[EPL_Q] * (dx * c + dy * s);
      b = -dx * s + dy * c;
      sa = rd[EPL_ZSX];
      sb = rd[EPL_ZSXI];
      ra = rd[EPL_ZRR];
      rb = rd[EPL_ZRRI];
    } else if constexpr (TYPE == LENSIM_NIE) {
      const double c = rd[NIE_C], s = rd[NIE_S];
      a = dx * c + dy * s;
      b = -dx * s + dy * c;
      sa = rd[NIE_XSX];
      sb = rd[NIE_YSX];
      ra = rd[NIE_XRR];
      rb = rd[NIE_YRR];
    } else {
      a = dx;
      b = dy;
      sa = st.sx[0];
      sb = st.sx[1];
      ra = st.rr[0];
      rb = st.rr[1];
    }
  }
  __device__ __forceinline__ void step() {
    a += sa;
    b += sb;
  }
  __device__ __forceinline__ void row() {
    a += ra;
    b += rb;
  }
};

// The exact position of sub-ray (sx, sy) of the pixel centred at (ra_c, dec_c).
struct SubRay {
  double ra_c, dec_c, o0, inv_s;
  int sx, sy;
  __device__ __forceinline__ void pos(const GridArgs &g, double &x, double &y) const {
    // the counters pass through readfirstlane (they are uniform), which keeps
    // the compiler from carrying them as float64 induction variables for
    // this rarely taken branch
    const double ox = o0 + __builtin_amdgcn_readfirstlane(sx) * inv_s;
    const double oy = o0 + __builtin_amdgcn_readfirstlane(sy) * inv_s;
    x = ra_c + g.m00 * ox + g.m01 * oy;
    y = dec_c + g.m10 * ox + g.m11 * oy;
  }
};

// beta -= alpha_scaling alpha of one compile-time deflector at its advanced
// coordinates; the EPL and SIE / NIE rotate back with (alpha_scaling cos phi,
// alpha_scaling sin phi) folded into the update.  An EPL sub-ray within 1e-12
// of the centre recomputes Z from its exact position (so that a ray exactly
// at the centre gets the reference's zero deflection, not the direction of
// the advanced coordinates' rounding).
template <typename T, int TYPE>
__device__ __forceinline__ void defl_fast(const Rec<T> &r, const T *coef_t, const double *coef_d,
                                          DeflCoords<TYPE> &u, double asc, const GridArgs &g, const SubRay &sr,
                                          double &bx, double &by) {
  if constexpr (TYPE == LENSIM_EPL) {
    double R2 = fma(u.a, u.a, u.b * u.b);
    if (R2 < 1e-24) {  // exact Z (the advance continues from it)
      double x, y;
      sr.pos(g, x, y);
      const double dx = x - r.d[R_CX], dy = y - r.d[R_CY];
      const double c = r.d[EPL_C], s = r.d[EPL_S];
      u.a = r.d[EPL_Q] * (dx * c + dy * s);
      u.b = -dx * s + dy * c;
      R2 = fma(u.a, u.a, u.b * u.b);
    }
    double fr, fi;
    if constexpr (sizeof(T) == sizeof(float))
      epl_major_f32(r, coef_t, coef_d, u.a, u.b, R2, fr, fi);
    else
      epl_major_f64(r, coef_d, u.a, u.b, R2, fr, fi);
    bx = fma(-r.d[EPL_AC], fr, fma(r.d[EPL_AS], fi, bx));
    by = fma(-r.d[EPL_AS], fr, fma(-r.d[EPL_AC], fi, by));
  } else if constexpr (TYPE == LENSIM_NIE) {
    double fx, fy;
    nie_major_dbl(r.d, u.a, u.b, fx, fy);
    bx = fma(-r.d[NIE_AC], fx, fma(r.d[NIE_AS], fy, bx));
    by = fma(-r.d[NIE_AS], fx, fma(-r.d[NIE_AC], fy, by));
  } else if constexpr (TYPE == LENSIM_NFW) {
    const double f = asc * nfw_factor_dbl(r.d, u.a, u.b);
    bx = fma(-f, u.a, bx);
    by = fma(-f, u.b, by);
  }
}

// The render for the common model families, the profile list fixed at compile
// time: deflector D0 (EPL, SIE / NIE or NFW) and optionally D1 (SHEAR, SIE /
// NIE or NFW; 0: none), in that order, then NSRC Sersic sources and NLL Sersic
// lens lights; one plane, no bulk list.  Per profile it is render_kernel's
// arithmetic, rearranged so that everything affine in the ray position is
// advanced by one addition per sub-ray instead of formed from the position:
// the deflectors' coordinates (DeflCoords), the lens lights' scaled
// elliptical coordinates, and w = theta - alpha_scaling alpha_SHEAR(theta)
// (the external shear is linear, so beta = w - alpha_scaling (alpha of the
// other deflectors)).  The records hold the steps (prepare_record's
// SubSteps).  In the float form each Sersic profile's values of a pixel are
// summed in float and multiplied by its amplitude in double at the end.
template <typename T, int D0, int D1, int NSRC, int NLL, bool KEEP>
__global__ __launch_bounds__(256) void render_fast_kernel(ModelArgs m, GridArgs g, const double *__restrict__ recd,
                                                          const float *__restrict__ recf,
                                                          const double *__restrict__ coefd,
                                                          const float *__restrict__ coeff, unsigned flags,
                                                          double *__restrict__ beta, T *__restrict__ out, float *__restrict__ blkmax) {
  constexpr bool kF32 = sizeof(T) == sizeof(float);
  static_assert(NSRC == 1, "the compile-time render takes one source");
  const int img = blockIdx.y;
  const int npix = g.nx * g.ny;
  const int pix0 = blockIdx.x * blockDim.x + threadIdx.x;
  const bool active = pix0 < npix;
  const int pix = active ? pix0 : npix - 1;  // inactive lanes stay for the wave reduction
  int i;
  const int j = div_by(pix, g.nx, g.inv_nx, i);
  const RecPtrs<T> rp = rec_ptrs<T>(m, recd, recf, coefd, coeff, img);
  constexpr int KS = D1 ? 2 : 1;  // first source record
  const Rec<T> r0{rp.recd, rp.rect};
  const Rec<T> r1{rp.recd + kRec, rp.rect + kRec};
  const size_t co = size_t(img) * m.n_epl * LENSIM_EPL_NMAX;  // D0's coefficients when it is the EPL (epl_index 0)
  // the pixel's first sub-ray (make_subgrid offsets, ImSim/Numerics/grid.py:60-62)
  const double ra_c = i * g.m00 + j * g.m01 + g.ra0;
  const double dec_c = i * g.m10 + j * g.m11 + g.dec0;
  const double inv_s = g.inv_s;
  const double o0 = g.o0;
  const double x0 = ra_c + g.m00 * o0 + g.m01 * o0;
  const double y0 = dec_c + g.m10 * o0 + g.m11 * o0;
  const bool do_src = (flags & LENSIM_IMAGE_SOURCE) && NSRC > 0;
  const bool do_light = (flags & LENSIM_IMAGE_LENS_LIGHT) && NLL > 0;
  const double asc = m.alpha_scaling;
  // w = theta - asc alpha_SHEAR(theta) and its steps
  double wx, wy, wsx, wsy, wrx, wry;
  if constexpr (D1 == LENSIM_SHEAR) {
    const double dx = x0 - r1.d[R_CX], dy = y0 - r1.d[R_CY];
    const double g1 = r1.d[SH_G1], g2 = r1.d[SH_G2];
    wx = x0 - asc * (g1 * dx + g2 * dy);
    wy = y0 - asc * (g2 * dx - g1 * dy);
    wsx = r1.d[SH_WSX];
    wsy = r1.d[SH_WSY];
    wrx = r1.d[SH_WRX];
    wry = r1.d[SH_WRY];
  } else {
    wx = x0;
    wy = y0;
    wsx = m.sub.sx[0];
    wsy = m.sub.sx[1];
    wrx = m.sub.rr[0];
    wry = m.sub.rr[1];
  }
  // relative to the source's centre, so beta - c_source comes out directly
  const double *rds = rp.recd + KS * kRec;
  wx -= rds[R_CX];
  wy -= rds[R_CY];
  // the Sersic floors: canonicalised once for the FP64 form's fmax, as float
  // bits for the float form's integer max
  const double umin_s = __builtin_canonicalize(rds[SE_UMIN]);
  const int uminb_s = __float_as_int(float(rds[SE_UMIN]));
  double umin_l[NLL > 0 ? NLL : 1];
  int uminb_l[NLL > 0 ? NLL : 1];
#pragma unroll
  for (int k = 0; k < NLL; ++k) {
    umin_l[k] = __builtin_canonicalize(rp.recd[(KS + NSRC + k) * kRec + SE_UMIN]);
    uminb_l[k] = __float_as_int(float(rp.recd[(KS + NSRC + k) * kRec + SE_UMIN]));
  }
  DeflCoords<D0> u0;
  u0.init(r0.d, m.sub, x0, y0);
  constexpr int D1C = (D1 == LENSIM_SHEAR || D1 == 0) ? LENSIM_NFW : D1;  // unused when D1 is SHEAR or none
  DeflCoords<D1C> u1;
  if constexpr (D1 == LENSIM_NIE || D1 == LENSIM_NFW) u1.init(r1.d, m.sub, x0, y0);
  // the lens lights' scaled elliptical coordinates
  double lx[NLL > 0 ? NLL : 1], ly[NLL > 0 ? NLL : 1];
#pragma unroll
  for (int k = 0; k < NLL; ++k) {
    const double *rd = rp.recd + (KS + NSRC + k) * kRec;
    const double dx = x0 - rd[R_CX], dy = y0 - rd[R_CY];
    lx[k] = fma(rd[SE_M00S], dx, rd[SE_M01S] * dy);
    ly[k] = fma(rd[SE_M01S], dx, rd[SE_M11S] * dy);
  }
  // per-profile sums of the Sersic values (float form) or the flux (FP64 form)
  float fs[NSRC > 0 ? NSRC : 1], fl[NLL > 0 ? NLL : 1];
#pragma unroll
  for (int k = 0; k < NSRC; ++k) fs[k] = 0.f;
#pragma unroll
  for (int k = 0; k < NLL; ++k) fl[k] = 0.f;
  double acc = 0.0;
  const bool eval = active && evaluated(g, i, j);
  for (int sy = 0; eval && sy < g.s; ++sy) {
    for (int sx = 0; sx < g.s; ++sx) {
      if (do_src) {
        const SubRay sr{ra_c, dec_c, o0, inv_s, sx, sy};
        double bx = wx, by = wy;
        defl_fast<T, D0>(r0, rp.coeft + co, rp.coefd + co, u0, asc, g, sr, bx, by);
        if constexpr (D1 == LENSIM_NIE || D1 == LENSIM_NFW)
          defl_fast<T, D1C>(r1, nullptr, nullptr, u1, asc, g, sr, bx, by);
        if constexpr (KEEP) {  // for the gradient's source launch (MpKeep)
          double *b = beta + ((size_t(img) * npix + pix) * size_t(g.s * g.s) + size_t(sy * g.s + sx)) * 2;
          AT(b, 0) = bx + rds[R_CX];
          AT(b, 1) = by + rds[R_CY];
        }
        // (bx, by) = beta - c_source
        const double xs = fma(rds[SE_M00S], bx, rds[SE_M01S] * by);
        const double ys = fma(rds[SE_M01S], bx, rds[SE_M11S] * by);
        if constexpr (kF32)
          fs[0] += sersic_u_f32(rds, reinterpret_cast<const float *>(rp.rect) + KS * kRec, xs, ys, uminb_s);
        else
          acc += rds[SE_AMP] * sersic_u_f64(rds, xs, ys, umin_s);
      }
      if (do_light) {
#pragma unroll
        for (int k = 0; k < NLL; ++k) {
          const double *rd = rp.recd + (KS + NSRC + k) * kRec;
          if constexpr (kF32)
            fl[k] += sersic_u_f32(rd, reinterpret_cast<const float *>(rp.rect) + (KS + NSRC + k) * kRec, lx[k],
                                  ly[k], uminb_l[k]);
          else
            acc += rd[SE_AMP] * sersic_u_f64(rd, lx[k], ly[k], umin_l[k]);
        }
      }
      // next sub-ray
      wx += wsx;
      wy += wsy;
      u0.step();
      if constexpr (D1 == LENSIM_NIE || D1 == LENSIM_NFW) u1.step();
#pragma unroll
      for (int k = 0; k < NLL; ++k) {
        const double *rd = rp.recd + (KS + NSRC + k) * kRec;
        lx[k] += rd[SE_XSX];
        ly[k] += rd[SE_YSX];
      }
    }
    // next row
    wx += wrx;
    wy += wry;
    u0.row();
    if constexpr (D1 == LENSIM_NIE || D1 == LENSIM_NFW) u1.row();
#pragma unroll
    for (int k = 0; k < NLL; ++k) {
      const double *rd = rp.recd + (KS + NSRC + k) * kRec;
      lx[k] += rd[SE_XRR];
      ly[k] += rd[SE_YRR];
    }
  }
  if constexpr (kF32) {
#pragma unroll
    for (int k = 0; k < NSRC; ++k) acc = fma(rp.recd[(KS + k) * kRec + SE_AMP], double(fs[k]), acc);
#pragma unroll
    for (int k = 0; k < NLL; ++k) acc = fma(rp.recd[(KS + NSRC + k) * kRec + SE_AMP], double(fl[k]), acc);
  }
  const T v = T(acc * (g.scale * m.flux_scaling));
  if (active) AT(out, size_t(img) * npix + pix) = v;
  if (blkmax) block_max_store(fabsf(float(v)), blkmax + size_t(img) * gridDim.x + blockIdx.x);
}

int check_launch(const char *where);

// The per-256-pixel block maxima of |image| that render_kernel stores for the
// MFMA convolution, from an image rendered by a kernel that keeps none.
template <typename T>
__global__ __launch_bounds__(256) void block_max_kernel(const T *__restrict__ v, int npix,
                                                        float *__restrict__ blkmax) {
  const int img = blockIdx.y;
  const int pix = blockIdx.x * blockDim.x + threadIdx.x;
  const float a = pix < npix ? fabsf(float(AT(v, size_t(img) * npix + pix))) : 0.f;
  block_max_store(a, blkmax + size_t(img) * gridDim.x + blockIdx.x);
}

// What a gradient keeps of its render for the adjoint kernels, so that the
// rays are not traced again: several planes, per ray and run the position, and
// beta; a bulk list that render_bulk_kernel takes, or in FP64 a model that
// render_fast_kernel takes, beta.
struct MpKeep {
  double4 *store;
  size_t per_img;
  void *beta;
};
int launch_mp_runs(const ModelArgs &m, int *tab, int n_img, hipStream_t st);
template <typename T>
int launch_render_mp(const ModelArgs &m, const GridArgs &g, const double *recd, const float *recf, const double *coefd,
                     const float *coeff, const int *tab, unsigned flags, const MpKeep &keep, T *out, int n_img,
                     hipStream_t st);

int bulk_classes(const ModelArgs &m, size_t npix);
template <typename T>
int launch_render_bulk(const ModelArgs &m, const GridArgs &g, const double *recd, const float *recf,
                       const double *coefd, const float *coeff, unsigned flags, const MpKeep &keep, T *out, int n_img,
                       hipStream_t st);

// Whether render_fast_kernel has the model (see launch_render); its deflectors.
template <typename T>
bool fast_model(const ModelArgs &m, unsigned flags, int &d0, int &d1) {
  auto sersic = [](int t) { return t == LENSIM_SERSIC || t == LENSIM_SERSIC_ELLIPSE; };
  auto nie = [](int t) { return t == LENSIM_SIE ? LENSIM_NIE : t; };
  bool fast = m.mp_n == 0 && m.n_bulk == 0 && (m.n_lens == 1 || m.n_lens == 2) && m.n_source == 1 &&
              (m.n_light == 0 || m.n_light == 1);
  d0 = d1 = 0;
  if (fast) {
    d0 = nie(m.types[0]);
    d1 = m.n_lens == 2 ? nie(m.types[1]) : 0;
    const bool pair = ((d0 == LENSIM_EPL || d0 == LENSIM_NIE || d0 == LENSIM_NFW) && (d1 == 0 || d1 == LENSIM_SHEAR)) ||
                      (d0 == LENSIM_NFW && d1 == LENSIM_NIE) || (d0 == LENSIM_NIE && d1 == LENSIM_NFW);
    fast = pair && (d0 != LENSIM_EPL || m.epl_index[0] == 0);
    // a light profile that a response column of the linear solve leaves out
    // (LENSIM_NULL) is no hindrance where nothing reads its record; in the
    // float form, whose two renders round differently, the columns stay with
    // render_kernel
    const bool f64 = sizeof(T) == sizeof(double);
    const int ts = m.types[m.n_lens], tl = m.n_light ? m.types[m.n_lens + 1] : LENSIM_NULL;
    fast = fast && (sersic(ts) || (f64 && ts == LENSIM_NULL && !(flags & LENSIM_IMAGE_SOURCE))) &&
           (sersic(tl) || m.n_light == 0 || (f64 && tl == LENSIM_NULL));
  }
  return fast;
}

// Launches render_fast_kernel when the model is one of its compile-time lists
// (EPL, SIE / NIE or NFW, each with or without SHEAR after it, NFW + SIE / NIE
// in either order; one Sersic source, none or one Sersic lens light),
// render_mp_kernel for several planes (tab: its plane runs),
// render_bulk_kernel for a bulk list over few pixels, else render_kernel.
template <typename T>
int launch_render(const ModelArgs &m, const GridArgs &g, const double *recd, const float *recf, const double *coefd,
                  const float *coeff, const int *tab, unsigned flags, const MpKeep &keep, T *out, float *blkmax,
                  int n_img, hipStream_t st) {
  const dim3 rgrid((g.nx * g.ny + 255) / 256, n_img);
  int d0, d1;
  const bool fast = fast_model<T>(m, flags, d0, d1);
  const bool share = !m.mp_n && (flags & LENSIM_IMAGE_SOURCE) && bulk_classes(m, size_t(g.nx) * g.ny) > 1;
  if (m.mp_n || share) {  // the block maxima for the MFMA convolution follow from the image in a second launch
    int rc = share ? launch_render_bulk<T>(m, g, recd, recf, coefd, coeff, flags, keep, out, n_img, st)
                   : launch_render_mp<T>(m, g, recd, recf, coefd, coeff, tab, flags, keep, out, n_img, st);
    if (rc || !blkmax) return rc;
    block_max_kernel<T><<<rgrid, 256, 0, st>>>(out, g.nx * g.ny, blkmax);
    return check_launch("block_max_kernel");
  }
  if (!fast) {
    // SIE / NIE and NFW deflect in double in the float form too; the kernel
    // is instantiated both ways so other models keep the float forms' registers
#define LENSIM_RENDER(H, D) \
  render_kernel<T, H, D><<<rgrid, 256, 0, st>>>(m, g, recd, recf, coefd, coeff, flags, out, blkmax)
    bool done = false;
    if constexpr (sizeof(T) == sizeof(float)) {
      if (m.has_nie_nfw) {
        if (m.has_halo) LENSIM_RENDER(true, true);
        else LENSIM_RENDER(false, true);
        done = true;
      }
    }
    if (!done) {
      if (m.has_halo) LENSIM_RENDER(true, false);
      else LENSIM_RENDER(false, false);
    }
#undef LENSIM_RENDER
    return check_launch("render_kernel");
  }
  const bool ll = m.n_light == 1 && m.types[m.n_lens + 1] != LENSIM_NULL;
  double *beta = sizeof(T) == sizeof(double) ? static_cast<double *>(keep.beta) : nullptr;
  auto launch = [&](auto kernel) {
    kernel<<<rgrid, 256, 0, st>>>(m, g, recd, recf, coefd, coeff, flags, beta, out, blkmax);
  };
#define LENSIM_FAST(A, B)                                                                             \
  do {                                                                                                \
    if constexpr (sizeof(T) == sizeof(double)) {                                                      \
      if (beta) {                                                                                     \
        launch(ll ? &render_fast_kernel<T, A, B, 1, 1, true> : &render_fast_kernel<T, A, B, 1, 0, true>); \
        break;                                                                                        \
      }                                                                                               \
    }                                                                                                 \
    launch(ll ? &render_fast_kernel<T, A, B, 1, 1, false> : &render_fast_kernel<T, A, B, 1, 0, false>); \
  } while (0)
  if (d0 == LENSIM_EPL && d1 == LENSIM_SHEAR) LENSIM_FAST(LENSIM_EPL, LENSIM_SHEAR);
  else if (d0 == LENSIM_EPL) LENSIM_FAST(LENSIM_EPL, 0);
  else if (d0 == LENSIM_NIE && d1 == LENSIM_SHEAR) LENSIM_FAST(LENSIM_NIE, LENSIM_SHEAR);
  else if (d0 == LENSIM_NIE && d1 == LENSIM_NFW) LENSIM_FAST(LENSIM_NIE, LENSIM_NFW);
  else if (d0 == LENSIM_NIE) LENSIM_FAST(LENSIM_NIE, 0);
  else if (d0 == LENSIM_NFW && d1 == LENSIM_SHEAR) LENSIM_FAST(LENSIM_NFW, LENSIM_SHEAR);
  else if (d0 == LENSIM_NFW && d1 == 0) LENSIM_FAST(LENSIM_NFW, 0);
  else LENSIM_FAST(LENSIM_NFW, LENSIM_NIE);
#undef LENSIM_FAST
  return check_launch("render_fast_kernel");
}

template <typename T, bool HALO, bool DBL>
__global__ __launch_bounds__(256) void raytrace_kernel(ModelArgs m, const double *__restrict__ recd,
                                                       const float *__restrict__ recf,
                                                       const double *__restrict__ coefd,
                                                       const float *__restrict__ coeff, const double *__restrict__ xs,
                                                       const double *__restrict__ ys, int64_t n_ray,
                                                       double *__restrict__ bx, double *__restrict__ by) {
  const int img = blockIdx.y;
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n_ray) return;
  const RecPtrs<T> rp = rec_ptrs<T>(m, recd, recf, coefd, coeff, img);
  double tx, ty;
  trace_ray<T, HALO, DBL, false>(m, rp, img, AT(xs, i), AT(ys, i), tx, ty);
  AT(bx, size_t(img) * n_ray + i) = tx;
  AT(by, size_t(img) * n_ray + i) = ty;
}

// A double moved across the lanes of each quad by a DPP quad permutation.
template <int CTRL>
__device__ __forceinline__ double dpp_quad_f64(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}

// The sum over the 4 lanes of a quad (every lane active), (v0 + v1) + (v2 + v3)
// in every lane: the additions commute exactly, so the four lanes hold the
// same bits.
__device__ __forceinline__ double quad_sum(double v) {
  v += dpp_quad_f64<0xB1>(v);  // quad_perm [1, 0, 3, 2]
  v += dpp_quad_f64<0x4E>(v);  // quad_perm [2, 3, 0, 1]
  return v;
}

// The sum over a wave (every lane active), uniform: the quads' sums, then
// the row's (row_ror 4 and 8 within each row of 16 lanes), then the four rows'
// sums read from their first lanes and added in order.
__device__ __forceinline__ double row_sum(double v) {  // over each row of 16 lanes, in all of them
  v = quad_sum(v);
  v += dpp_quad_f64<0x124>(v);  // row_ror:4
  v += dpp_quad_f64<0x128>(v);  // row_ror:8
  return v;
}
__device__ __forceinline__ double wave_sum(double v) {
  v = row_sum(v);
  auto row = [&](int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
  };
  return (row(0) + row(16)) + (row(32) + row(48));
}

// ---- several planes ----
// Deflectors on one plane follow each other in the plane order with T_ij = 0
// between them: the ray does not move across them and they all deflect it at
// one position.  A run is up to kMpRun consecutive planes with one position,
// T_z and reduced-to-physical factor; it is the unit the kernels below work in.
constexpr int kMpRun = 64;
constexpr int kMpPrep = 1024;

struct MpTab {  // see mp_tab_ints
  const int *start, *run_of, *plane_of, *who;
  int n, dup, sub;
};
static_assert(LENSIM_CONVERGENCE < 128, "a deflector's type shares an int with its index");
constexpr int kWhoBits = 24;

__host__ __device__ constexpr bool sub_type(int t) {  // add_deflection's SUB
  return t == LENSIM_NULL || t == LENSIM_TNFW || t == LENSIM_SHEAR || t == LENSIM_CONVERGENCE;
}
__device__ __forceinline__ MpTab mp_tab(const ModelArgs &m, const int *__restrict__ tab, int img) {
  const int *t = tab + (m.mp_stride ? size_t(img) * mp_tab_ints(m) : 0);
  CHECK_SPAN(t, size_t(mp_tab_ints(m)) * sizeof(int));
  return MpTab{t + 3,    t + 3 + m.mp_n, t + 2 + 2 * m.mp_n, t + 2 + 2 * m.mp_n + m.n_defl, t[0],
               t[1], t[2]};
}

// The runs of one set of plane arrays, by a block of NT threads: every thread
// takes a contiguous piece of the planes; a maximum scan over the pieces gives
// the plane the position last changed at, and so the planes that start a run
// (there, and every kMpRun planes after), a sum scan their numbers.
template <int NT>
__device__ __forceinline__ void mp_runs_block(const ModelArgs &m, int *__restrict__ tab_all, int set) {
  int *tab = tab_all + size_t(set) * mp_tab_ints(m);
  const size_t o = size_t(set) * size_t(m.mp_stride);
  const int nd = m.mp_n - 1, t = threadIdx.x, per = (nd + NT - 1) / NT;
  const int q0 = min(nd, t * per), q1 = min(nd, q0 + per);
  int *start = tab + 3, *run_of = tab + 3 + m.mp_n, *plane_of = tab + 2 + 2 * m.mp_n;
  int *who = plane_of + m.n_defl;
  auto moved = [&](int q) {
    return q == 0 || AT(m.mp_tij, o + q) != 0.0 || AT(m.mp_tz, o + q) != AT(m.mp_tz, o + q - 1) ||
           AT(m.mp_r2p, o + q) != AT(m.mp_r2p, o + q - 1);
  };
  __shared__ int sc[2][NT];
  __shared__ int dup, other;
  auto scan = [&](int v, auto op) {  // inclusive, over the threads
    sc[0][t] = v;
    __syncthreads();
    int b = 0;
    for (int d = 1; d < NT; d <<= 1, b ^= 1) {
      sc[b ^ 1][t] = t >= d ? op(sc[b][t], sc[b][t - d]) : sc[b][t];
      __syncthreads();
    }
    const int r = sc[b][t];
    const int before = t ? sc[b][t - 1] : -1;
    __syncthreads();
    return make_int2(r, before);
  };
  int last = -1;
  for (int q = q0; q < q1; ++q)
    if (moved(q)) last = q;
  const int from = scan(last, [](int a, int b) { return a > b ? a : b; }).y;
  int at = from, cnt = 0;
  for (int q = q0; q < q1; ++q) {
    if (moved(q)) at = q;
    cnt += (q - at) % kMpRun == 0;
  }
  const int2 s = scan(cnt, [](int a, int b) { return a + b; });
  int idx = t ? s.y : 0;
  at = from;
  for (int q = q0; q < q1; ++q) {
    if (moved(q)) at = q;
    if ((q - at) % kMpRun == 0) AT(start, idx++) = q;
    AT(run_of, q) = idx - 1;
  }
  for (int k = t; k < m.n_defl; k += NT) AT(plane_of, k) = -1;
  if (t == 0) dup = other = 0;
  __syncthreads();
  for (int k = t; m.n_bulk > 0 && !m.bulk_type && k < m.n_bulk; k += NT)
    if (!sub_type(AT(m.bulk_types, k))) other = 1;
  for (int q = q0; q < q1; ++q) {
    int k = AT(m.mp_order, q);
    k = k < 0 ? 0 : (k >= m.n_defl ? m.n_defl - 1 : k);  // a bad index cannot read outside the records
    if (atomicExch(&AT(plane_of, k), q) >= 0) dup = 1;
    int type = k < m.n_lens ? m.types[k] : (m.bulk_type ? m.bulk_type : AT(m.bulk_types, k - m.n_lens));
    if (k >= m.n_lens && !bulk_type_ok_dev(type)) type = LENSIM_NULL;
    AT(who, q) = k | type << kWhoBits;
  }
  __syncthreads();
  if (t == NT - 1) {
    AT(start, s.x) = nd;
    AT(tab, 0) = s.x;
    AT(tab, 1) = dup;
    AT(tab, 2) = !other;
  }
}
__global__ __launch_bounds__(1024) void mp_runs_kernel(ModelArgs m, int *__restrict__ tab_all) {
  mp_runs_block<1024>(m, tab_all, blockIdx.x);
}

int launch_mp_runs(const ModelArgs &m, int *tab, int n_img, hipStream_t st) {
  mp_runs_kernel<<<(unsigned)mp_tab_sets(m, n_img), 1024, 0, st>>>(m, tab);
  return check_launch("mp_runs_kernel");
}

// The sums of (vx, vy) over the block's waves (eight at most), lane by lane and
// in wave order, in every wave.  buf alternates between consecutive calls, so
// that no barrier is needed before the write.
constexpr int kSumWaves = 8;
struct WaveSums {
  double2 part[2][kSumWaves][65];  // (rows of 64 measured 2% slower on 16 images of 300^2 and 1000 subhalos)
};
__device__ __forceinline__ void across_waves(WaveSums &red, int buf, int nw, double &vx, double &vy) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  red.part[buf][wave][lane] = double2{vx, vy};
  __syncthreads();
  vx = vy = 0.0;
  for (int w = 0; w < nw; ++w) {
    const double2 v = red.part[buf][w][lane];
    vx += v.x;
    vy += v.y;
  }
}

// Classes that a run's deflectors are summed in (every classes-th of them, then
// the classes): their number follows the image's rays and the list's length
// alone, and with it the order of the sums, whatever launch does them
// (mp_launch).  Measured: a line of sight of 5256 0.46 ms with 16, 0.52 with 8 for
// 100^2 rays, 2.95 with 8, 4.2 with 16 for 400^2; 48 halos on 8 planes 10% more
// with 4 than with 8 at 100^2 x 4 rays, the same or up to 30% less at 180^2 x 9;
// 8 halos on 2 planes, 30 on 10 4 to 10% less.  Past 2^28 rays two, which keeps a
// launch's threads below 2^32.
__host__ __device__ inline int mp_classes(int n_defl, int64_t n_ray, bool sub) {
  if (n_ray > (int64_t(1) << 28)) return 2;
  if (n_defl >= 1024) return sub && n_ray < 65536 ? 16 : 8;
  return n_defl > 32 && n_ray < 24576 ? 8 : 4;
}

// A wave of a multi-plane kernel and the 64 rays it holds.  The waves of a block
// share their rays and take a class of a run each; SOLO: a block is one wave, which takes
// the classes in turn, without a barrier.
template <bool SOLO>
struct MpWave {
  int wave, nw, classes;
  __device__ __forceinline__ explicit MpWave(int classes)
      : wave(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)), nw(int(blockDim.x) >> 6), classes(classes) {}
  __device__ __forceinline__ bool lead() const { return SOLO || wave == 0; }  // loads, adds and stores for the rays
  __device__ __forceinline__ void barrier() const {
    if constexpr (!SOLO) __syncthreads();
  }
};
template <bool SOLO>
struct MpRed {
  double2 part[2][16][65];  // rows of 65: the 16 values of a ray lie on distinct banks
  double2 sum[2][64];
};
template <>
struct MpRed<true> {};

// (vx, vy): the sum over a run's `len` members of what one(q, vx, vy) adds for
// member q, in every wave that holds the rays.  buf alternates between
// consecutive calls, so that no barrier is needed before the write.  Up to eight
// classes are added in class order, each wave reading all of them; sixteen in
// the order of row_sum (the quads of classes in pairs, (Q0 + Q3) + (Q2 + Q1)):
// sixteen waves would each read 16 KB of LDS (2000 cycles a call), so there a
// row of 16 lanes sums one ray's values and every wave reads the sums, at the
// price of a second barrier.
template <bool SUB, typename F>
__device__ __forceinline__ void run_sum(const MpWave<false> &w, MpRed<false> &red, int buf, int len, double &vx, double &vy,
                                        F one) {
  const int lane = threadIdx.x & 63;
  double ax = 0.0, ay = 0.0;
  for (int q = w.wave; q < len; q += w.nw) one(q, ax, ay);
  // (by the lane's own index: by w.wave rays of 1828 halos over 202^2 took 662 us for 652)
  red.part[buf][threadIdx.x >> 6][lane] = double2{ax, ay};
  __syncthreads();
  if (SUB && w.nw == 16) {
    const int ray = threadIdx.x >> 4, c = threadIdx.x & 15;
    const double2 v = red.part[buf][c][ray];
    const double2 s{row_sum(v.x), row_sum(v.y)};
    if (c == 0) red.sum[buf][ray] = s;
    __syncthreads();
    vx = red.sum[buf][lane].x;
    vy = red.sum[buf][lane].y;
    return;
  }
  vx = vy = 0.0;
  for (int c = 0; c < w.nw; ++c) {
    const double2 v = red.part[buf][c][lane];
    vx += v.x;
    vy += v.y;
  }
}
// (Up to three members: their sum in order is that of either tree.)
template <bool SUB, typename F>
__device__ __forceinline__ void run_sum(const MpWave<true> &w, MpRed<true> &, int, int len, double &vx, double &vy, F one) {
  const bool tree = SUB && w.classes == 16 && len > 3;
  const int nt = tree ? 16 : min(len, w.classes);
  double ax = 0.0, ay = 0.0, bx = 0.0, by = 0.0, dx = 0.0, dy = 0.0;  // a pair, a quad, Q0 + Q3
  vx = vy = 0.0;
  for (int t = 0; t < nt; ++t) {
    const int c = !tree ? t : (t < 4 ? t : (t < 8 ? t + 8 : (t < 12 ? t : t - 8)));
    double sx = 0.0, sy = 0.0;
    for (int q = c; q < len; q += w.classes) one(q, sx, sy);
    if (!tree) {
      vx += sx;
      vy += sy;
      continue;
    }
    ax = t & 1 ? ax + sx : sx;
    ay = t & 1 ? ay + sy : sy;
    if (!(t & 1)) continue;
    bx = t & 2 ? bx + ax : ax;
    by = t & 2 ? by + ay : ay;
    if (t == 3) dx = bx, dy = by;
    if (t == 7) dx += bx, dy += by;
    if (t == 11) vx = bx, vy = by;
    if (t == 15) vx = dx + (vx + bx), vy = dy + (vy + by);
  }
}

// Multi-plane ray tracing (MultiPlaneBulk.ray_shooting,
// LensModel/MultiPlane/multi_plane_bulk.py:152-212) of 64 rays, one per lane.
// A run's deflectors are the same for all lanes of a wave (a record comes by
// scalar loads) and 1 / T_z is taken once per run.  Shared by the block's waves,
// the chain of record loads and deflections a ray waits for is as many times
// shorter as the runs are long: one lane per ray left 400^2 rays through 5256
// deflectors at 2.4 waves per SIMD, waiting on memory for most of a deflector's
// 1100 cycles.  Runs of a deflector or two, or rays enough to fill the chip,
// gain nothing by it and pay a barrier per run: solo (mp_shape).  Every thread
// of a block that shares reaches this call.
// each(c, x, y): run c's position, for callers that keep it.
template <typename T, bool HALO, bool DBL, bool DBL_TNFW, bool SUB, bool SOLO, typename F>
__device__ __forceinline__ void block_trace(const ModelArgs &m, const RecPtrs<T> &rp, const MpTab &tab,
                                            const double *__restrict__ tij, const double *__restrict__ tzs,
                                            const double *__restrict__ r2p, int img, double x, double y,
                                            const MpWave<SOLO> &w, MpRed<SOLO> &red, double &bx, double &by, F each) {
  const int lane = threadIdx.x & 63;
  double angx = x, angy = y, px = 0.0, py = 0.0;
  // the deflectors of a run, a lane each, loaded one run ahead
  auto members = [&](int p0, int p1) { return p0 + lane < p1 ? AT(tab.who, p0 + lane) : 0; };
  int p0 = 0, p1 = tab.n ? AT(tab.start, 1) : 0;
  int ks = members(p0, p1);
  double dt = AT(tij, 0), itz = rcp_full(AT(tzs, 0)), f = AT(r2p, 0);
  for (int c = 0; c < tab.n; ++c) {
    const int p2 = c + 1 < tab.n ? AT(tab.start, c + 2) : p1;
    const int ks_next = members(p1, p2);
    const double dt_next = AT(tij, p1), tz_next = AT(tzs, p1), f_next = AT(r2p, p1);  // p1 <= nd: the source's plane
    px = fma(angx, dt, px);
    py = fma(angy, dt, py);
    const double xr = px * itz, yr = py * itz;
    each(c, xr, yr);
    double ax, ay;
    run_sum<SUB>(w, red, c & 1, p1 - p0, ax, ay, [&](int q, double &sx, double &sy) {
      const int k = __builtin_amdgcn_readlane(ks, q);
      deflect_one<T, HALO, DBL, DBL_TNFW, SUB>(m, rp, img, k & ((1 << kWhoBits) - 1), k >> kWhoBits, xr, yr, sx, sy);
    });
    angx = fma(-ax, f, angx);
    angy = fma(-ay, f, angy);
    p0 = p1;
    p1 = p2;
    ks = ks_next;
    dt = dt_next;
    itz = rcp_full(tz_next);
    f = f_next;
  }
  px = fma(angx, dt, px);  // the source's plane
  py = fma(angy, dt, py);
  bx = px * itz;
  by = py * itz;
}

// The plane arrays of image img as restrict pointers.
#define LENSIM_MP_ARRAYS(m, img)                                        \
  const size_t mp_o = size_t(img) * size_t((m).mp_stride);              \
  const double *tij = (m).mp_tij + mp_o, *tzs = (m).mp_tz + mp_o, *r2p = (m).mp_r2p + mp_o

// A launch over `some` of n_ray rays of n_img images: a wave per class, or solo.
// Sharing gains where the runs are long and the chip is not full: solo are lists
// of less than two deflectors a run (by the caller's bound, at least a run per
// deflector without one), and from 4096 waves of rays (16 a CU; 2048 for lists
// whose types take twice the registers) runs of less than four turns of the
// classes.  Against a wave per class, and one lane per ray or quad over the whole
// list before (us a call, FP64 images): seven deflectors on seven planes, 16 of
// 180^2 x 9 rays 342, 2740, 335; 16 halos on one plane, one of 100^2 x 4 rays
// 87, 37, 46, 32 of them 185, 225, 257; 40 of several types on 5 planes 16 of
// 180^2 x 9 2000, 3880, 2450.
struct MpLaunch {
  bool solo;
  unsigned threads;
  dim3 grid;
};
MpLaunch mp_launch(const ModelArgs &m, size_t n_ray, size_t some, int n_img, bool sub) {
  const int classes = mp_classes(m.n_defl, int64_t(n_ray), sub);
  const size_t groups = (some + 63) / 64, all = groups * n_img;
  MpLaunch l;
  l.solo = m.n_defl < 2 * m.mp_runs || (all >= 2048 && !sub) ||
           (all >= 4096 && m.n_defl < 4 * int64_t(classes) * m.mp_runs);
  l.threads = l.solo ? 64 : 64 * classes;
  l.grid = dim3((unsigned)groups, n_img);
  return l;
}

// Threads a block of a multi-plane kernel may have.
constexpr int mp_threads_most(bool sub, bool solo) { return solo ? 64 : (sub ? 1024 : 512); }
// Waves per SIMD the solo render is held to (its FP64 form without halos keeps
// three so, as render_kernel's; the others would spill or have them anyway).
template <typename T>
constexpr int mp_render_waves(bool halo, bool solo) {
  return sizeof(T) == sizeof(double) && !halo && solo ? 3 : 1;
}

template <typename T, bool HALO, bool DBL, bool SUB, bool SOLO>
__global__ __launch_bounds__(mp_threads_most(SUB, SOLO)) void raytrace_mp_kernel(ModelArgs m, const double *__restrict__ recd,
                                                           const float *__restrict__ recf,
                                                           const double *__restrict__ coefd,
                                                           const float *__restrict__ coeff,
                                                           const int *__restrict__ tab_all,
                                                           const double *__restrict__ xs,
                                                           const double *__restrict__ ys, int64_t n_ray,
                                                           int64_t first, bool both,
                                                           double *__restrict__ bx, double *__restrict__ by) {
  __shared__ MpRed<SOLO> red;
  const int img = blockIdx.y;
  const int64_t ray0 = first + int64_t(blockIdx.x) * 64 + (threadIdx.x & 63);
  const bool active = ray0 < n_ray;
  const int64_t ray = active ? ray0 : n_ray - 1;  // lanes past the end follow the last ray
  const RecPtrs<T> rp = rec_ptrs<T>(m, recd, recf, coefd, coeff, img);
  const MpTab tab = mp_tab(m, tab_all, img);
  if (both && bool(tab.sub) != SUB) return;  // the other instantiation's launch takes it
  const MpWave<SOLO> w(mp_classes(m.n_defl, n_ray, SUB));
  LENSIM_MP_ARRAYS(m, img);
  double tx, ty;
  block_trace<T, HALO, DBL, false, SUB, SOLO>(m, rp, tab, tij, tzs, r2p, img, AT(xs, ray), AT(ys, ray), w, red, tx, ty,
                                              [](int, double, double) {});
  if (active && w.lead()) {
    AT(bx, size_t(img) * n_ray + ray) = tx;
    AT(by, size_t(img) * n_ray + ray) = ty;
  }
}

// Rays a round takes of image img's adjoint store, from its runs (all of them
// where there is no deflector and so nothing to store).
__device__ __forceinline__ int64_t round_rays(size_t per_img, int runs) {
  return runs > 0 ? int64_t(per_img / size_t(runs) / 64 * 64) : int64_t(1) << 31;
}

// render_kernel for several planes: the block's waves walk the sub-rays of its
// 64 pixels together (block_trace); the first wave adds the light and stores.
template <typename T, bool HALO, bool DBL, bool SUB, bool SOLO>
__global__ __launch_bounds__(mp_threads_most(SUB, SOLO))
__attribute__((amdgpu_waves_per_eu(mp_render_waves<T>(HALO, SOLO)))) void render_mp_kernel(ModelArgs m, GridArgs g, const double *__restrict__ recd,
                                                         const float *__restrict__ recf,
                                                         const double *__restrict__ coefd,
                                                         const float *__restrict__ coeff,
                                                         const int *__restrict__ tab_all, unsigned flags, bool both,
                                                         MpKeep keep, T *__restrict__ out) {
  __shared__ MpRed<SOLO> red;
  const int img = blockIdx.y;
  const int npix = g.nx * g.ny;
  const int pix0 = int(blockIdx.x * 64) + int(threadIdx.x & 63);
  const bool active = pix0 < npix;
  const int pix = active ? pix0 : npix - 1;
  int i;
  const int j = div_by(pix, g.nx, g.inv_nx, i);
  const RecPtrs<T> rp = rec_ptrs<T>(m, recd, recf, coefd, coeff, img);
  const MpTab tab = mp_tab(m, tab_all, img);
  if (both && bool(tab.sub) != SUB) return;  // the other instantiation's launch takes it
  const MpWave<SOLO> w(mp_classes(m.n_defl, npix, SUB));
  LENSIM_MP_ARRAYS(m, img);
  const double ra_c = i * g.m00 + j * g.m01 + g.ra0;
  const double dec_c = i * g.m10 + j * g.m11 + g.dec0;
  const bool do_src = (flags & LENSIM_IMAGE_SOURCE) && m.n_source > 0;
  const bool do_light = (flags & LENSIM_IMAGE_LENS_LIGHT) && m.n_light > 0;
  const int k_src0 = m.n_defl, k_src1 = m.n_defl + m.n_source, k_l1 = m.n_prof;
  double acc = 0.0;
  const bool eval = active && evaluated(g, i, j);
  const bool any = __any(eval);  // the same in every wave that holds the pixels
  const int64_t cap = keep.store ? round_rays(keep.per_img, tab.n) : 0;
  const bool keeps = active && w.lead() && cap >= int64_t(npix) * g.s * g.s;
  for (int sy = 0; any && sy < g.s; ++sy) {
    const double oy = g.o0 + sy * g.inv_s;
    for (int sx = 0; sx < g.s; ++sx) {
      const double ox = g.o0 + sx * g.inv_s;
      const double x = ra_c + g.m00 * ox + g.m01 * oy;
      const double y = dec_c + g.m10 * ox + g.m11 * oy;
      double bx = x, by = y;
      if (do_src) {
        w.barrier();  // the last sub-ray's sums are read
        const size_t ray = size_t(pix) * (g.s * g.s) + size_t(sy * g.s + sx);
        block_trace<T, HALO, DBL, DBL, SUB, SOLO>(
            m, rp, tab, tij, tzs, r2p, img, x, y, w, red, bx, by, [&](int c, double xr, double yr) {
              if (keeps) AT(keep.store, size_t(img) * keep.per_img + ray + size_t(c) * cap) = double4{xr, yr, 0.0, 0.0};
            });
        if (keeps && keep.beta) {
          T *b = static_cast<T *>(keep.beta) + (size_t(img) * npix * size_t(g.s * g.s) + ray) * 2;
          AT(b, 0) = T(bx);
          AT(b, 1) = T(by);
        }
      }
      if (eval && w.lead()) {
        if (do_src) acc += light_sum<T>(m, rp, k_src0, k_src1, bx, by);
        if (do_light) acc += light_sum<T>(m, rp, k_src1, k_l1, x, y);
      }
    }
  }
  const T v = T(acc * (g.scale * m.flux_scaling));
  if (active && w.lead()) AT(out, size_t(img) * npix + pix) = v;
}

// Whether every deflector is a subhalo or linear (add_deflection's SUB): 1
// yes, 0 no, 2 when only the device knows (bulk deflectors of several types:
// both instantiations are launched then, and mp_runs_kernel's flag ends one).
int sub_list(const ModelArgs &m) {
  for (int k = 0; k < m.n_lens; ++k)
    if (!sub_type(m.types[k])) return 0;
  if (m.n_bulk == 0) return 1;
  return m.bulk_type ? int(sub_type(m.bulk_type)) : 2;
}

template <typename T>
int launch_render_mp(const ModelArgs &m, const GridArgs &g, const double *recd, const float *recf, const double *coefd,
                     const float *coeff, const int *tab, unsigned flags, const MpKeep &keep, T *out, int n_img,
                     hipStream_t st) {
  const size_t npix = size_t(g.nx) * g.ny;
  const int sub = sub_list(m);
  auto launch = [&](auto kernel, const MpLaunch &l) {
    kernel<<<l.grid, l.threads, 0, st>>>(m, g, recd, recf, coefd, coeff, tab, flags, sub == 2, keep, out);
  };
#define LENSIM_RENDER(H, D, S)                                                                          \
  do {                                                                                                  \
    const MpLaunch l = mp_launch(m, npix, npix, n_img, S);                                              \
    launch(l.solo ? &render_mp_kernel<T, H, D, S, true> : &render_mp_kernel<T, H, D, S, false>, l);     \
  } while (0)
  // the float form deflects SIE / NIE and the NFW family in double
  constexpr bool kF32 = sizeof(T) == sizeof(float);
  if (sub) LENSIM_RENDER(true, kF32, true);
  if (sub != 1) {
    if (kF32 && m.has_nie_nfw && m.has_halo) LENSIM_RENDER(true, kF32, false);
    else if (kF32 && m.has_nie_nfw) LENSIM_RENDER(false, kF32, false);
    else if (m.has_halo) LENSIM_RENDER(true, false, false);
    else LENSIM_RENDER(false, false, false);
  }
#undef LENSIM_RENDER
  return check_launch("render_mp_kernel");
}

// render_kernel for a bulk list over few pixels: the block's waves hold the
// same 64 pixels and share the list (the first takes the inline deflectors
// too), their sums meeting in LDS once per sub-ray; the first adds the light.
// A lane per pixel alone leaves 4 images of 100^2 at less than one wave per
// SIMD, each waiting out 200 deflectors' latency four times over (479 us; 275
// so, and the adjoint kernel's 204 us of deflections fall away with the beta
// kept here: a gradient 989 -> 605 us).  Where the pixels fill the chip by
// themselves the shared form idles seven waves of eight through the light and
// waits at its barriers (64 halos, 128 images of 150^2 in mixed form 2.2 -> 2.9
// ms against render_kernel):
// SOLO: a block is one wave, which takes the classes in turn and adds them in the
// same order (2.1 ms).  beta: see MpKeep.
template <typename T, bool HALO, bool DBL, bool SOLO>
__global__ __launch_bounds__(SOLO ? 64 : 512) void render_bulk_kernel(ModelArgs m, GridArgs g, const double *__restrict__ recd,
                                                          const float *__restrict__ recf,
                                                          const double *__restrict__ coefd,
                                                          const float *__restrict__ coeff, unsigned flags,
                                                          int classes, T *__restrict__ beta, T *__restrict__ out) {
  __shared__ std::conditional_t<SOLO, char, WaveSums> red;
  const int img = blockIdx.y, nw = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int npix = g.nx * g.ny;
  const int pix0 = blockIdx.x * 64 + (threadIdx.x & 63);
  const bool active = pix0 < npix;
  const int pix = active ? pix0 : npix - 1;
  int i;
  const int j = div_by(pix, g.nx, g.inv_nx, i);
  const RecPtrs<T> rp = rec_ptrs<T>(m, recd, recf, coefd, coeff, img);
  const double ra_c = i * g.m00 + j * g.m01 + g.ra0;
  const double dec_c = i * g.m10 + j * g.m11 + g.dec0;
  const bool do_light = (flags & LENSIM_IMAGE_LENS_LIGHT) && m.n_light > 0;
  const int k_src0 = m.n_defl, k_src1 = m.n_defl + m.n_source, k_l1 = m.n_prof;
  double acc = 0.0;
  const bool eval = active && evaluated(g, i, j);
  const bool any = __any(eval);  // the same in every wave: they hold the same pixels
  const int rays = any ? g.s * g.s : 0;
  for (int r = 0; r < rays; ++r) {
    const int sy = r / g.s, sx = r - sy * g.s;
    const double oy = g.o0 + sy * g.inv_s, ox = g.o0 + sx * g.inv_s;
    const double x = ra_c + g.m00 * ox + g.m01 * oy;
    const double y = dec_c + g.m10 * ox + g.m11 * oy;
    double ax = 0.0, ay = 0.0;
    if (wave == 0)
      for (int k = 0; k < m.n_lens; ++k) deflect_one<T, HALO, DBL>(m, rp, img, k, m.types[k], x, y, ax, ay);
    if constexpr (SOLO) {
      double tx = 0.0, ty = 0.0;
      for (int c = 0; c < classes; ++c) {
        deflect_bulk<T, HALO, DBL>(m, rp, x, y, ax, ay, c, classes);
        tx += ax;
        ty += ay;
        ax = ay = 0.0;
      }
      ax = tx;
      ay = ty;
    } else {
      deflect_bulk<T, HALO, DBL>(m, rp, x, y, ax, ay, wave, nw);
      across_waves(red, r & 1, nw, ax, ay);
    }
    if (wave == 0 && eval) {
      const double bx = x - ax * m.alpha_scaling, by = y - ay * m.alpha_scaling;
      if (beta) {
        T *b = beta + ((size_t(img) * npix + pix) * size_t(g.s * g.s) + size_t(r)) * 2;
        AT(b, 0) = T(bx);
        AT(b, 1) = T(by);
      }
      acc += light_sum<T>(m, rp, k_src0, k_src1, bx, by);
      if (do_light) acc += light_sum<T>(m, rp, k_src1, k_l1, x, y);
    }
  }
  if (active && wave == 0) AT(out, size_t(img) * npix + pix) = T(acc * (g.scale * m.flux_scaling));
}

// Classes that a bulk list is summed in (every classes-th deflector, then the
// classes) by render_bulk_kernel, 1 for render_kernel: as many waves for one
// image as put four on each SIMD while each takes eight deflectors or more.
// They depend on the image alone (not on the batch), as the order of the sums
// does.  Measured with 1 / 2 / 4 / 8 waves: 16 mixed images of 300^2 and 1000
// subhalos 21.8 / 21.5 / 20.95 / 22.2 ms a call, 4 gradients of 100^2 and 200 in
// FP64 1010 / 684 / 605 / 604 us.
int bulk_classes(const ModelArgs &m, size_t npix) {
  int nw = 1;
  while (m.mp_n == 0 && m.n_source > 0 && nw < 8 && npix * nw < 64 * 4096 && m.n_bulk >= 16 * nw) nw *= 2;
  return nw;
}

// Whether a gradient's render_bulk_kernel keeps beta for bulk_adjoint_kernel:
// not where the float form renders in double what the adjoint takes in float.
template <typename T>
bool bulk_keeps(const ModelArgs &m, size_t npix) {
  return bulk_classes(m, npix) > 1 && (sizeof(T) == sizeof(double) || !m.has_nie_nfw);
}

template <typename T>
int launch_render_bulk(const ModelArgs &m, const GridArgs &g, const double *recd, const float *recf,
                       const double *coefd, const float *coeff, unsigned flags, const MpKeep &keep, T *out, int n_img,
                       hipStream_t st) {
  const size_t npix = size_t(g.nx) * g.ny;
  const dim3 grid((unsigned)((npix + 63) / 64), n_img);
  const int classes = bulk_classes(m, npix);
  // Solo where the pixels' waves alone are one and a half times what the chip
  // holds (2 a SIMD of the forms that deflect in double, 4 of the float one; of
  // the float form's long lists, whose last waves leave the chip idle longer,
  // eight times).  Shared against solo: 64 halos in FP64, 16 images of 100^2 x 4
  // rays 350, 372 us, 32 of them 677, 562, 128 of 150^2 5530, 4120; in mixed form
  // 223, 273, 407, 417, 2910, 2140; 1000 in mixed form, 16 of 300^2 x 9 30.2, 30.9
  // ms, 128 of 150^2 x 4 33.7, 30.9.
  const size_t waves = (npix + 63) / 64 * n_img;
  const bool dbl = sizeof(T) == sizeof(double) || m.has_nie_nfw;
  const bool solo = waves >= (dbl ? 3072 : (m.n_bulk < 512 ? 6144 : 32768));
  auto launch = [&](auto kernel) {
    kernel<<<grid, solo ? 64 : 64 * classes, 0, st>>>(m, g, recd, recf, coefd, coeff, flags, classes,
                                                      static_cast<T *>(keep.beta), out);
  };
#define LENSIM_RENDER(H, D) launch(solo ? &render_bulk_kernel<T, H, D, true> : &render_bulk_kernel<T, H, D, false>)
  constexpr bool kF32 = sizeof(T) == sizeof(float);  // as render_kernel's
  if (kF32 && m.has_nie_nfw && m.has_halo) LENSIM_RENDER(true, kF32);
  else if (kF32 && m.has_nie_nfw) LENSIM_RENDER(false, kF32);
  else if (m.has_halo) LENSIM_RENDER(true, false);
  else LENSIM_RENDER(false, false);
#undef LENSIM_RENDER
  return check_launch("render_bulk_kernel");
}

// raytrace_mp_kernel's launches for a call, in pieces of 2^28 rays (a launch's
// threads stay below 2^32).
template <typename T>
int launch_raytrace_mp(const ModelArgs &m, const double *recd, const float *recf, const double *coefd,
                       const float *coeff, const int *tab, const double *x, const double *y, int64_t n_ray, int n_img,
                       double *bx, double *by, hipStream_t st) {
  const int sub = sub_list(m);
  constexpr bool kF32 = sizeof(T) == sizeof(float);
  constexpr int64_t kPiece = int64_t(1) << 28;
  for (int64_t r0 = 0; r0 < n_ray; r0 += kPiece) {
    const int64_t nr = n_ray - r0 < kPiece ? n_ray - r0 : kPiece;
    auto launch = [&](auto kernel, const MpLaunch &l) {
      kernel<<<l.grid, l.threads, 0, st>>>(m, recd, recf, coefd, coeff, tab, x, y, n_ray, r0, sub == 2, bx, by);
    };
#define LENSIM_TRACE(H, D, S)                                                                           \
  do {                                                                                                  \
    const MpLaunch l = mp_launch(m, size_t(n_ray), size_t(nr), n_img, S);                               \
    launch(l.solo ? &raytrace_mp_kernel<T, H, D, S, true> : &raytrace_mp_kernel<T, H, D, S, false>, l); \
  } while (0)
    // the float form keeps the float TNFW of a list without SIE / NIE or NFW
    // (rays within 2e-6 of FP64); those deflect in double (see nie_defl)
    if (sub) LENSIM_TRACE(true, false, true);
    if (sub != 1) {
      if (kF32 && m.has_nie_nfw && m.has_halo) LENSIM_TRACE(true, kF32, false);
      else if (kF32 && m.has_nie_nfw) LENSIM_TRACE(false, kF32, false);
      else if (m.has_halo) LENSIM_TRACE(true, false, false);
      else LENSIM_TRACE(false, false, false);
    }
#undef LENSIM_TRACE
    const int rc = check_launch("raytrace_mp_kernel");
    if (rc) return rc;
  }
  return LENSIM_OK;
}

template <typename T>
__global__ __launch_bounds__(256) void light_kernel(ModelArgs m, const double *__restrict__ recd,
                                                    const float *__restrict__ recf, int k0, int k1,
                                                    const double *__restrict__ xs, const double *__restrict__ ys,
                                                    int64_t n_ray, double *__restrict__ flux) {
  const int img = blockIdx.y;
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n_ray) return;
  const RecPtrs<T> rp = rec_ptrs<T>(m, recd, recf, nullptr, nullptr, img);
  AT(flux, size_t(img) * n_ray + i) = light_sum<T>(m, rp, k0, k1, AT(xs, i), AT(ys, i));
}

struct ConvArgs {
  int nx, ny, kx, ky, kyp, edge, n_tiles_x;  // kyp: kernel height padded to kWin
  const double *data, *noise, *expo, *mask;
  double exposure_time, bkg2;
  double inv_t;  // 1 / exposure_time, formed on the host
  void *gout;  // optional dlogL/dmodel per pixel (compute type)
  int64_t dstride;  // data / noise elements between batch images (0: shared)
};


// d logL / d model of one pixel: logL = -1/2 mask (m - d)^2 / V(m) with
// V = max(m, 0)/t + bkg^2 (dV/dm = 1/t for m >= 0, the branch the reference's
// jnp.where(data >= 0, ...) takes) or the noise map's square (dV/dm = 0).
__device__ __forceinline__ double dlogl_dm(const ConvArgs &c, size_t p, double m, int img) {
  const size_t q = p + size_t(img) * size_t(c.dstride);  // per-image observation
  const double d = AT(c.data, q);
  double var, dvar;
  if (c.noise) {
    var = AT(c.noise, q) * AT(c.noise, q);
    dvar = 0.0;
  } else {
    const double it = c.expo ? rcp_refined(AT(c.expo, p)) : c.inv_t;  // 1 / exposure
    var = fma(m >= 0.0 ? m : 0.0, it, c.bkg2);
    dvar = m >= 0.0 ? it : 0.0;
  }
  const double r = (m - d) * rcp_refined(var);
  double gp = -(r - 0.5 * r * r * dvar);
  if (c.mask) gp *= AT(c.mask, p);
  return gp;
}

template <typename T>
__device__ __forceinline__ double chi2_pixel(const ConvArgs &c, size_t p, T model_t, int img) {
  const size_t q = p + size_t(img) * size_t(c.dstride);  // per-image observation
  const double m = double(model_t);
  const double d = AT(c.data, q);
  double var;
  if (c.noise) {
    const double nm = AT(c.noise, q);
    var = nm * nm;
  } else {
    const double it = c.expo ? rcp_refined(AT(c.expo, p)) : c.inv_t;  // 1 / exposure
    const double mpos = (m >= 0.0) ? m : 0.0;
    var = fma(mpos, it, c.bkg2);
  }
  double chi = (m - d) * (m - d) * rcp_refined(var);
  if (c.mask) chi *= AT(c.mask, p);
  return chi;
}

// The chi^2 partial of 32 x 16 pixels, tile (txi, ty) of the image, by a wave: v
// is lane l's sum of eight consecutive rows of column l % 32, in row order.
__device__ __forceinline__ void tile_partial(const ConvArgs &c, double v, int lane, int img, int txi, int ty,
                                             double *partial) {
  v = wave_sum(v);
  const int n = c.n_tiles_x * ((c.ny + 15) >> 4);
  if (lane == 0 && 16 * ty < c.ny) AT(partial, size_t(img) * n + ty * c.n_tiles_x + txi) = v;
}

// out[y][x] = sum_{a,c} in[y - cy + a][x - cx + c] * Kf[a][c]  (Kf = flipped kernel).
// Block = TX columns x (TY / kWin) row groups; each thread computes kWin
// consecutive rows of one column from a register window that slides down the
// LDS tile, so consecutive lanes read consecutive LDS words.
// LW: the weights are staged in LDS behind the tile.  For launches of fewer
// blocks than CUs: there each step's scalar loads of the weights would miss
// the caches in turn (the kernel was just written by another launch), one
// memory latency per step.
// CLS: 0, or conv_f64_kernel's classes of kernel columns for the same bits as
// its (the columns class by class, the classes' sums in order) and its chi^2
// partials.
template <typename T, int TY, bool LW, int CLS>
__global__ __launch_bounds__(256) void conv_kernel(ConvArgs c, const T *__restrict__ in,
                                                   const double *__restrict__ kt, T *__restrict__ out,
                                                   double *__restrict__ partial) {
  constexpr int TX = ConvTile<T>::TX, NT = TX * TY / kWin;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *tile = reinterpret_cast<T *>(smem_raw);
  const int img = blockIdx.y;
  const int tile_id = blockIdx.x;
  const int tyi = tile_id / c.n_tiles_x, txi = tile_id - tyi * c.n_tiles_x;
  const int y0 = tyi * TY, x0 = txi * TX;
  const int cy = (c.ky - 1) / 2, cx = (c.kx - 1) / 2;
  const int kyp = c.kyp;
  const int TH = TY + kyp - 1, TW = TX + c.kx - 1;
  const int THp = TH | 1;  // column stride of the column-major tile: odd, so lanes hit distinct banks
  const T *src = in + size_t(img) * c.nx * c.ny;
  const int tid = threadIdx.x;
  // kLd elements per thread and pass: all their loads are issued before the
  // first LDS store waits, so a launch of few blocks (LW) pays one memory
  // latency per pass rather than one per element.  Large launches hide that
  // latency across blocks and keep one element per pass (eight measured
  // slower for the float adjoint convolution of the gradient).
  constexpr int kLd = LW ? 8 : 1;
  for (int base = tid; base < TH * TW; base += NT * kLd) {
    T v[kLd];
    int at[kLd];
#pragma unroll
    for (int u = 0; u < kLd; ++u) {
      const int idx = base + u * NT;
      const int ly = idx / TW, lx = idx - ly * TW;
      int gy = y0 - cy + ly, gx = x0 - cx + lx;
      v[u] = T(0);
      at[u] = idx < TH * TW ? lx * THp + ly : -1;
      if (idx >= TH * TW || ly >= TY + c.ky - 1) {
        // past the tile, or rows that only meet the zero padding of the kernel height
      } else if (c.edge) {
        gy = gy < 0 ? 0 : (gy >= c.ny ? c.ny - 1 : gy);
        gx = gx < 0 ? 0 : (gx >= c.nx ? c.nx - 1 : gx);
        v[u] = AT(src, gy * c.nx + gx);
      } else if (gy >= 0 && gy < c.ny && gx >= 0 && gx < c.nx) {
        v[u] = AT(src, gy * c.nx + gx);
      }
    }
#pragma unroll
    for (int u = 0; u < kLd; ++u)
      if (at[u] >= 0) tile[at[u]] = v[u];
  }
  const int nch = kyp / kWin, nsteps = c.kx * nch;
  double *wl = reinterpret_cast<double *>(smem_raw + ((size_t(THp) * TW * sizeof(T) + 7) & ~size_t(7)));
  if constexpr (LW) {
    for (int idx = tid; idx < nsteps * kWin; idx += NT) wl[idx] = AT(kt, idx);
  } else {
    CHECK_SPAN(kt, size_t(nsteps + 1) * kWin * sizeof(double));
  }
  __syncthreads();
  const int lx = tid % TX, tg = tid / TX;
  // float64 accumulation in both forms (full-rate FMA on CDNA4)
  double acc[kWin], sum[kWin];  // sum: of the classes before
#pragma unroll
  for (int r = 0; r < kWin; ++r) acc[r] = sum[r] = 0.0;
  // steps t = (kernel column cc, row chunk ch) flattened; the window of step
  // t + 1 is loaded while step t is computed
  const T *colbase = tile + lx * THp + tg * kWin;
  double buf[2 * kWin - 1];
#pragma unroll
  for (int q = 0; q < 2 * kWin - 1; ++q) buf[q] = double(colbase[q]);
  double w[kWin];
#pragma unroll
  for (int jj = 0; jj < kWin; ++jj) w[jj] = LW ? wl[jj] : kt[jj];
  int cc = 0, ch = 0;
  for (int t = 0; t < nsteps; ++t) {
    bool next_class = false;
    if (++ch == nch) {
      ch = 0;
      if (CLS > 1) {
        next_class = cc + CLS >= c.kx;
        cc = next_class ? cc % CLS + 1 : cc + CLS;
      } else {
        ++cc;
      }
    }
    // next step's weights and window are requested before this step's FMAs
    // (the compiler still waits for them before the FMAs: the weights are
    // scalar loads, which complete out of order, so any wait on the shared
    // counter is a wait for all of them; latency is hidden across waves)
    double wn[kWin];
    T nb[2 * kWin - 1];
    if (t + 1 < nsteps) {
      if constexpr (LW) {
#pragma unroll
        for (int jj = 0; jj < kWin; ++jj) wn[jj] = wl[cc * kyp + ch * kWin + jj];
      } else {
        const double *kw = kt + cc * kyp + ch * kWin;
#pragma unroll
        for (int jj = 0; jj < kWin; ++jj) wn[jj] = kw[jj];
      }
      const T *col = colbase + cc * THp + ch * kWin;
#pragma unroll
      for (int q = 0; q < 2 * kWin - 1; ++q) nb[q] = col[q];
    }
#pragma unroll
    for (int jj = 0; jj < kWin; ++jj) {
#pragma unroll
      for (int r = 0; r < kWin; ++r) acc[r] = fma(buf[r + jj], w[jj], acc[r]);
    }
#pragma unroll
    for (int q = 0; q < 2 * kWin - 1; ++q) buf[q] = double(nb[q]);
#pragma unroll
    for (int jj = 0; jj < kWin; ++jj) w[jj] = wn[jj];
    if (next_class) {
#pragma unroll
      for (int r = 0; r < kWin; ++r) {
        sum[r] += acc[r];
        acc[r] = 0.0;
      }
    }
  }
  const int x = x0 + lx;
  double chi = 0.0;
  if (x < c.nx) {
#pragma unroll
    for (int r = 0; r < kWin; ++r) {
      const int y = y0 + tg * kWin + r;
      if (y < c.ny) {
        const size_t p = size_t(y) * c.nx + x;
        const T m = T(CLS > 1 ? sum[r] : acc[r]);
        if (out) AT(out, size_t(img) * c.nx * c.ny + p) = m;
        if (partial) chi += chi2_pixel<T>(c, p, m, img);
        if (c.gout) AT(static_cast<T *>(c.gout), size_t(img) * c.nx * c.ny + p) = T(dlogl_dm(c, p, double(m), img));
      }
    }
  }
  if (partial && CLS) {
    tile_partial(c, chi, tid & 63, img, txi, (y0 >> 4) + (tid >> 6), partial);
  } else if (partial) {
    // wave reduction then one value per wave through LDS (fixed order)
    for (int off = 32; off > 0; off >>= 1) chi += __shfl_xor(chi, off, 64);
    __syncthreads();
    double *red = reinterpret_cast<double *>(smem_raw);
    const int wave = tid >> 6, lane = tid & 63;
    if (lane == 0) red[wave] = chi;
    __syncthreads();
    if (tid == 0) {
      double s = 0.0;
      for (int w = 0; w < NT / 64; ++w) s += red[w];
      AT(partial, size_t(img) * gridDim.x + tile_id) = s;
    }
  }
}


// The FP64 form's convolution: conv_kernel's sum on a tile of 32 columns x 2 R H
// rows.  Each of the 4 H waves takes the kernel columns of one class (mod 4) for
// 32 x 2 R pixels; the classes' sums meet in LDS and are added in class order,
// so that neither the sum nor the chi^2 partials (of 32 x 16 pixels) depend on
// the block's shape, which follows the batch.  A lane has R consecutive rows of
// one column: of a kernel column it reads each image value once (consecutive
// lanes, consecutive words) and holds 24 of them in three groups of eight that
// rotate by name, so that no register is moved.  GW: the weights by scalar
// loads, else from LDS (few blocks: there every step's loads would miss the
// caches in turn).  The FP64 vector unit has the matrix unit's rate here, and no
// band of zeros to multiply (a Toeplitz block on v_mfma_f64_16x16x4 spends 41 of
// 56 columns at 41 x 41).  Measured: 71^2 with 21 x 21 22.3 -> 7.4 us, 60^2 with
// 11 x 11 13.6 -> 6.2, 4 images of 100^2 with 21 x 21 30 -> 9, 64 of 180^2 with 41
// x 41 184 -> 165 (42 TFLOP/s of the 65 a matrix product reaches; the rest is
// the ragged edge tiles, 13%, halo loads and each column's first reads).
template <int R, int H, int CLS, bool GW>
__global__ __launch_bounds__(64 * CLS * H) void conv_f64_kernel(ConvArgs c, int th, const double *__restrict__ in,
                                                       const double *__restrict__ kt, double *__restrict__ out,
                                                       double *__restrict__ partial) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double *tile = reinterpret_cast<double *>(smem_raw);
  int img = blockIdx.y, tile_id = blockIdx.x;
  {  // XCD-aware order, as conv_mfma_kernel
    const int n_blk = gridDim.x * gridDim.y, lin = blockIdx.y * gridDim.x + blockIdx.x;
    if ((n_blk & 7) == 0) {
      const int logical = (lin & 7) * (n_blk >> 3) + (lin >> 3);
      img = logical / gridDim.x;
      tile_id = logical - img * gridDim.x;
    }
  }
  const int tyi = tile_id / c.n_tiles_x, txi = tile_id - tyi * c.n_tiles_x;
  const int y0 = tyi * 2 * R * H, x0 = txi * 32;
  const int cy = (c.ky - 1) / 2, cx = (c.kx - 1) / 2;
  const int TH = 2 * R * H + c.ky - 1, TW = 32 + c.kx - 1;
  const double *src = in + size_t(img) * c.nx * c.ny;
  const int tid = threadIdx.x;
  double *wl = tile + conv_f64_tile(c.kx, th, R, H, CLS);
  static_assert(R % CLS == 0 && R * H % 8 == 0, "");
  // the weights and the tile, eight loads in flight per thread: every thread
  // loads (from the nearest pixel of the image), zeros are chosen afterwards
  constexpr int NT = 64 * CLS * H, kLd = 8, kLw = 2;
  const int nt = TH * TW, nwt = c.kx * c.kyp;
  const int dy = NT / TW, dx = NT - dy * TW;
  double w0[kLw];
  if constexpr (GW) CHECK_SPAN(kt, size_t(nwt) * sizeof(double));
#pragma unroll
  for (int u = 0; u < kLw; ++u) w0[u] = GW ? 0.0 : AT(kt, min(tid + u * NT, nwt - 1));
  int ly = tid / TW, lx0 = tid - ly * TW;
  auto some = [&](auto n, int base) {
    constexpr int kN = decltype(n)::value;
    double v[kN];
    bool ok[kN];
#pragma unroll
    for (int u = 0; u < kN; ++u) {
      const int gy = y0 - cy + ly, gx = x0 - cx + lx0;
      const int py = min(max(gy, 0), c.ny - 1), px = min(max(gx, 0), c.nx - 1);
      v[u] = AT(src, py * c.nx + px);
      ok[u] = c.edge || (py == gy && px == gx);
      lx0 += dx;
      ly += dy;
      const bool wrap = lx0 >= TW;
      lx0 -= wrap ? TW : 0;
      ly += wrap;
    }
#pragma unroll
    for (int u = 0; u < kN; ++u)
      if (base + tid + u * NT < nt) tile[base + tid + u * NT] = ok[u] ? v[u] : 0.0;
  };
  int base = 0;
  for (; base + (kLd - 2) * NT < nt; base += NT * kLd) some(std::integral_constant<int, kLd>(), base);
  for (; base < nt; base += NT * 2) some(std::integral_constant<int, 2>(), base);
#pragma unroll
  for (int u = 0; u < kLw; ++u)
    if (!GW && tid + u * NT < nwt) wl[tid + u * NT] = w0[u];
  for (int at = tid + kLw * NT; !GW && at < nwt; at += NT * kLd) {
    double v[kLd];
#pragma unroll
    for (int u = 0; u < kLd; ++u) v[u] = AT(kt, min(at + u * NT, nwt - 1));
#pragma unroll
    for (int u = 0; u < kLd; ++u)
      if (at + u * NT < nwt) wl[at + u * NT] = v[u];
  }
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lx = lane & 31;
  const int cls = wave % CLS, row0 = wave / CLS * 2 * R + (lane >> 5) * R;  // the lane's first row of the tile
  double acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = 0.0;
  for (int cc = cls; cc < c.kx; cc += CLS) {
    const double *col = tile + row0 * TW + lx + cc;
    const double *w = (GW ? kt : wl) + cc * c.kyp;
    double g0[8], g1[8], g2[8];
    auto load = [&](double (&g)[8]) {
#pragma unroll
      for (int i = 0; i < 8; ++i) g[i] = col[i * TW];
      col += 8 * TW;
    };
    // the next n taps of w: tap u reads rows u .. u + R - 1 of a, b, d
    auto taps = [&](auto n, const double (&a)[8], const double (&b)[8], const double (&d)[8]) {
#pragma unroll
      for (int u = 0; u < decltype(n)::value; ++u) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int q = u + r;
          acc[r] = fma(q < 8 ? a[q & 7] : (q < 16 ? b[q & 7] : d[q & 7]), w[u], acc[r]);
        }
      }
      w += 8;
    };
    // a kernel has an odd number of rows: 1, 3, 5 or 7 in its last group
    auto tail = [&](int n, const double (&a)[8], const double (&b)[8], const double (&d)[8]) {
      if (n & 4) {
        if (n & 2) taps(std::integral_constant<int, 7>(), a, b, d);
        else taps(std::integral_constant<int, 5>(), a, b, d);
      } else {
        if (n & 2) taps(std::integral_constant<int, 3>(), a, b, d);
        else taps(std::integral_constant<int, 1>(), a, b, d);
      }
    };
    constexpr std::integral_constant<int, 8> k8;
    load(g0);
    load(g1);
    if (R + c.ky - 1 > 16) load(g2);
    int left = c.ky;
    while (true) {
      if (left < 8) {
        tail(left, g0, g1, g2);
        break;
      }
      taps(k8, g0, g1, g2);
      load(g0);
      if ((left -= 8) < 8) {
        tail(left, g1, g2, g0);
        break;
      }
      taps(k8, g1, g2, g0);
      load(g1);
      if ((left -= 8) < 8) {
        tail(left, g2, g0, g1);
        break;
      }
      taps(k8, g2, g0, g1);
      load(g2);
      left -= 8;
    }
  }
  if constexpr (CLS > 1) {
    __syncthreads();  // the tile is read: the classes' sums take its place
#pragma unroll
    for (int r = 0; r < R; ++r) tile[(wave * R + r) * 64 + lane] = acc[r];
    __syncthreads();
  }
  const int x = x0 + lx;
  double chi[R / CLS];
#pragma unroll
  for (int i = 0; i < R / CLS; ++i) {
    const int r = cls + CLS * i, y = y0 + row0 + r;
    double m = acc[i];
    if constexpr (CLS > 1) {
      const double *s = tile + (wave / CLS * CLS * R + r) * 64 + lane;
      m = ((s[0] + s[R * 64]) + s[2 * R * 64]) + s[3 * R * 64];
    }
    chi[i] = 0.0;
    if (x < c.nx && y < c.ny) {
      const size_t p = size_t(y) * c.nx + x;
      if (out) AT(out, size_t(img) * c.nx * c.ny + p) = m;
      if (partial) chi[i] = chi2_pixel<double>(c, p, m, img);
      if (c.gout) AT(static_cast<double *>(c.gout), size_t(img) * c.nx * c.ny + p) = dlogl_dm(c, p, m, img);
    }
  }
  if (partial) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < R / CLS; ++i) tile[(row0 + cls + CLS * i) * 32 + lx] = chi[i];
    __syncthreads();
    for (int q = wave; q < R * H / 8; q += CLS * H) {
      double v = 0.0;
#pragma unroll
      for (int i = 0; i < 8; ++i) v += tile[(q * 16 + (lane >> 5) * 8 + i) * 32 + lx];
      tile_partial(c, v, lane, img, txi, (y0 >> 4) + q, partial);
    }
  }
}

// ------------------------------------------------ MFMA convolution (mixed) --
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// B fragments of the banded kernel rows, in the lane layout of
// v_mfma_f32_16x16x32_f16 (lane l holds B[8 (l / 16) + j][l % 16], j < 8),
// split into fp16 hi + lo of the kernel scaled by 2^sk (max |K| 2^sk in
// [2^14, 2^15)).  One thread per fragment; every block reduces the kernel
// maximum itself (K is small), block 0 stores sk in hdr[0].  The fragments of
// the padding steps (ky * nks up to n_steps) are zero.
// One 256-thread block (index b) of the fragment preparation.
__device__ void psf_mfma_prep_block(const double *__restrict__ k, int kx, int ky, int nks, int n_steps,
                                    int *__restrict__ hdr, half8 *__restrict__ frag, int b) {
  __shared__ double red[4];
  double m = 0.0;
  for (int i = threadIdx.x; i < kx * ky; i += blockDim.x) m = fmax(m, fabs(AT(k, i)));
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  const double mx = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
  const int sk = (mx > 0.0 && isfinite(mx)) ? 14 - ilogb(mx) : 0;
  if (b == 0 && threadIdx.x == 0) AT(hdr, 0) = sk;
  const double scale = ldexp(1.0, sk);  // exact power of two
  const int idx = b * 256 + threadIdx.x;
  if (idx >= n_steps * 2 * 64) return;
  const int lane = idx & 63, s = (idx >> 6) & 1, ak = idx >> 7;
  if (ak >= ky * nks) {
    AT(frag, idx) = half8{};
    return;
  }
  const int a = ak / nks, ks = ak - a * nks;
  const int n = lane & 15, g = lane >> 4;
  const double *krow = k + size_t(ky - 1 - a) * kx;
  half8 v;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int c = 32 * ks + 8 * g + j - n;  // tap of the flipped kernel row a
    const double w = (c >= 0 && c < kx) ? AT(krow, kx - 1 - c) * scale : 0.0;
    const _Float16 h = (_Float16)w;
    v[j] = s == 0 ? h : (_Float16)(w - (double)h);
  }
  AT(frag, idx) = v;
}

__global__ __launch_bounds__(256) void psf_mfma_prep_kernel(const double *__restrict__ k, int kx, int ky, int nks,
                                                            int n_steps, int *__restrict__ hdr,
                                                            half8 *__restrict__ frag) {
  psf_mfma_prep_block(k, kx, ky, nks, n_steps, hdr, frag, blockIdx.x);
}

// The PSF preparation of a call, folded into the record preparation's launch
// (the two are independent): mode 1 the flipped transposed kernel, 2 the MFMA
// fragments.
struct PsfJob {
  int mode;
  const double *k;
  int kx, ky, kyp, nks, n_steps;
  double *kt;
  int *hdr;
  half8 *frag;
};

int psf_job_blocks(const PsfJob &pj) {
  if (pj.mode == 1) return (pj.kyp * pj.kx + 255) / 256;
  if (pj.mode == 2) return (pj.n_steps * 2 * 64 + 255) / 256;
  return 0;
}

// Blocks [0, nb_prep): one thread per (image, profile) record; [nb_prep, nb_prep
// + nb_runs): a set of plane runs each; the rest: the PSF job.
__global__ __launch_bounds__(256) void prep_psf_kernel(ModelArgs m, const double *__restrict__ params, int n_img,
                                                       double *__restrict__ recd, float *__restrict__ recf,
                                                       double *__restrict__ coefd, float *__restrict__ coeff,
                                                       double *__restrict__ dcoefd, float *__restrict__ dcoeff,
                                                       PsfJob pj, int *__restrict__ tab, int nb_prep, int nb_runs) {
  if (int(blockIdx.x) < nb_prep) {
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx < n_img * m.n_prof) prep_one(m, params, n_img, idx, recd, recf, coefd, coeff, dcoefd, dcoeff);
    return;
  }
  if (int(blockIdx.x) < nb_prep + nb_runs) {
    mp_runs_block<256>(m, tab, blockIdx.x - nb_prep);
    return;
  }
  const int b = blockIdx.x - nb_prep - nb_runs;
  if (pj.mode == 2) {
    psf_mfma_prep_block(pj.k, pj.kx, pj.ky, pj.nks, pj.n_steps, pj.hdr, pj.frag, b);
  } else {
    const int idx = b * 256 + threadIdx.x;
    if (idx < pj.kyp * pj.kx) psf_prep_one(pj.k, pj.kx, pj.ky, pj.kyp, pj.kt, 1, idx);
  }
}

// Direct 'same' convolution on the matrix cores: block = 64 rows x 16 TL
// columns (4 waves x TL tiles of 16 x 16; NKS K-steps of 32 per kernel row).
// The padded tile sits in LDS as fp16 hi and lo planes of the image scaled by
// 2^sa (sa from the per-image max); per kernel row a and K-step, three MFMAs
// (hi.hi, hi.lo, lo.hi) accumulate in float32, and the float sums are folded
// into float64 accumulators once per unrolled body of rows.
template <int NKS, int TL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 3))) void conv_mfma_kernel(
    ConvArgs c, int ls, const float *__restrict__ in,
                                                        const int *__restrict__ hdr,
                                                        const half8 *__restrict__ frag,
                                                        const float *__restrict__ blkmax, int nblk,
                                                        float *__restrict__ out, double *__restrict__ partial) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  // XCD-aware order: consecutive workgroups go to different XCDs (round
  // robin over 8), so the workgroups one XCD receives are given consecutive
  // (image, tile) indices and share their halos in that XCD's L2
  int img = blockIdx.y, tile_id = blockIdx.x;
  {
    const int n_blk = gridDim.x * gridDim.y, lin = blockIdx.y * gridDim.x + blockIdx.x;
    if ((n_blk & 7) == 0) {
      const int logical = (lin & 7) * (n_blk >> 3) + (lin >> 3);
      img = logical / gridDim.x;
      tile_id = logical - img * gridDim.x;
    }
  }
  const int tyi = tile_id / c.n_tiles_x, txi = tile_id - tyi * c.n_tiles_x;
  const int Y0 = tyi * kMfTY, X0 = txi * 16 * TL;
  const int cy = (c.ky - 1) / 2, cx = (c.kx - 1) / 2;
  const int TH = kMfTY + c.ky - 1, TW = 16 * (TL - 1) + 32 * NKS;
  _Float16 *lh = reinterpret_cast<_Float16 *>(smem_raw);
  _Float16 *ll = lh + TH * ls;
  const int tid = threadIdx.x;
  const float *src = in + size_t(img) * c.nx * c.ny;
  // the wave index is the same on every lane: read it as a scalar, so the
  // tile rows a wave loads are addressed with scalar, not vector, arithmetic
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 15, lg = lane >> 4;
  // The padded tile: each wave fills rows wave, wave + 4, ..., lanes along a
  // row, in batches of kLdRows rows x kLdCols 64-column chunks.  Every load
  // reads a clamped (in-image) address and is zeroed after the fact outside
  // the image, so a whole batch is issued before the first load is waited
  // for; the first batch is in flight while the image maximum is reduced.
  constexpr int kLdRows = 8, kLdCols = (16 * (TL - 1) + 32 * NKS + 63) / 64;
  float v[kLdRows][kLdCols];
  auto load_batch = [&](int ly0) {
#pragma unroll
    for (int r = 0; r < kLdRows; ++r) {
      const int gy0 = Y0 - cy + ly0 + kMfWaves * r;
      const int gy = gy0 < 0 ? 0 : (gy0 >= c.ny ? c.ny - 1 : gy0);
      const bool row_ok = c.edge || gy0 == gy;
#pragma unroll
      for (int q = 0; q < kLdCols; ++q) {
        const int gx0 = X0 - cx + 64 * q + lane;
        const int gx = gx0 < 0 ? 0 : (gx0 >= c.nx ? c.nx - 1 : gx0);
        const float x = AT(src, size_t(gy) * c.nx + gx);
        v[r][q] = (row_ok && (c.edge || gx0 == gx)) ? x : 0.f;
      }
    }
  };
  load_batch(wave);
  // image max |value| from the render blocks' maxima
  __shared__ float smax[4];
  {
    float mv = 0.f;
    for (int b = tid; b < nblk; b += 256) mv = fmaxf(mv, AT(blkmax, size_t(img) * nblk + b));
    for (int off = 32; off > 0; off >>= 1) mv = fmaxf(mv, __shfl_xor(mv, off, 64));
    if ((tid & 63) == 0) smax[tid >> 6] = mv;
    __syncthreads();
  }
  const float mx = fmaxf(fmaxf(smax[0], smax[1]), fmaxf(smax[2], smax[3]));
  const int sa = (mx > 0.f && isfinite(mx)) ? 14 - ilogbf(mx) : 0;
  const int sk = AT(hdr, 0);
  const float scale_a = ldexpf(1.0f, sa);  // exact power of two
  auto store_batch = [&](int ly0) {
#pragma unroll
    for (int r = 0; r < kLdRows; ++r) {
      const int ly = ly0 + kMfWaves * r;
#pragma unroll
      for (int q = 0; q < kLdCols; ++q) {
        const int lx = 64 * q + lane;
        if (lx < TW && ly < TH) {
          const float xs = v[r][q] * scale_a;
          const _Float16 h = (_Float16)xs;
          lh[ly * ls + lx] = h;
          ll[ly * ls + lx] = (_Float16)(xs - (float)h);
        }
      }
    }
  };
  store_batch(wave);
  for (int ly0 = wave + kMfWaves * kLdRows; ly0 < TH; ly0 += kMfWaves * kLdRows) {
    load_batch(ly0);
    store_batch(ly0);
  }
  __syncthreads();
  double dacc[TL][4];
#pragma unroll
  for (int t = 0; t < TL; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) dacc[t][j] = 0.0;
  const int rowbase = (16 * wave + li) * ls + 8 * lg;
  // One step per (kernel row a, K block ks).  The rows are padded with
  // zero-B rows to a multiple of U; a body covers U rows (R = U * NKS steps).
  // Two register sets of B fragments (from L2) alternate between bodies: a
  // set is refilled with the steps 2R ahead as soon as its body's MFMAs are
  // issued, so its loads fly during the other set's body.  No load sits under
  // a branch (the refills past the last step re-read the last fragments and
  // are not used).  The float sums are folded into the float64 accumulators
  // once per pair of bodies (2U kernel rows).
  constexpr int U = mfma_unroll(NKS), R = U * NKS;
  const int ky_pad = (c.ky + U - 1) / U * U, n_steps = ky_pad * NKS;
  half8 bq[2][R][2];
  // The fragments are read as a buffer (resource in scalar registers): the
  // step's offset is a scalar and the lane's a fixed vector offset, so a load
  // needs no vector address arithmetic.  Reads past the n_steps fragments
  // (none are issued) would return zeros.
  const __amdgpu_buffer_rsrc_t frs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<half8 *>(frag), (short)0, n_steps * 2048, 0x00020000);
  const int voff = lane * 16;
  CHECK_SPAN(frag, size_t(n_steps) * 2048);
  auto refill = [&](half8 (&b)[R][2], int s0) {
#pragma unroll
    for (int p = 0; p < R; ++p) {
      const int q = __builtin_amdgcn_readfirstlane(s0 + p < n_steps ? s0 + p : n_steps - 1);
      b[p][0] = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(frs, voff, q * 2048, 0));
      b[p][1] = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(frs, voff, q * 2048 + 1024, 0));
    }
  };
  floatx4 acc[TL];
  auto zero = [&]() {
#pragma unroll
    for (int t = 0; t < TL; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  };
  auto fold = [&]() {
#pragma unroll
    for (int t = 0; t < TL; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) dacc[t][j] += double(acc[t][j]);
  };
  auto body = [&](const half8 (&b)[R][2], int a0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int ar = a0 + u < c.ky ? a0 + u : c.ky - 1;  // padding rows re-read the last row (times zero B)
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        const int p = u * NKS + ks;
        half8 ah[TL], al[TL];
#pragma unroll
        for (int t = 0; t < TL; ++t) {
          const int off = rowbase + ar * ls + 16 * t + 32 * ks;
          ah[t] = *reinterpret_cast<const half8 *>(lh + off);
          al[t] = *reinterpret_cast<const half8 *>(ll + off);
        }
#pragma unroll
        for (int t = 0; t < TL; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[t], b[p][0], acc[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < TL; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[t], b[p][1], acc[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < TL; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[t], b[p][0], acc[t], 0, 0, 0);
      }
    }
  };
  refill(bq[0], 0);
  refill(bq[1], R);
  int a0 = 0;
  for (; a0 + 2 * U <= ky_pad; a0 += 2 * U) {
    zero();
    body(bq[0], a0);
    refill(bq[0], (a0 + 2 * U) * NKS);
    body(bq[1], a0 + U);
    refill(bq[1], (a0 + 3 * U) * NKS);
    fold();
  }
  if (a0 < ky_pad) {  // an odd number of bodies: the last one
    zero();
    body(bq[0], a0);
    fold();
  }
  // lane l holds D[4 (l / 16) + j][l % 16] of each tile
  const double unscale = ldexp(1.0, -(sa + sk));
  // chi^2: one partial per 16 x 16 output tile, at [img][tile row][tile
  // column] of the image's 16 x 16 tiling, so the order of the sum does not
  // depend on the block width (which the plan picks by batch size): a request
  // has the same log-likelihood in any batch
  const int n16x = (c.nx + 15) >> 4, n16 = n16x * ((c.ny + 15) >> 4);
  const int ty16 = (Y0 >> 4) + wave;
#pragma unroll
  for (int t = 0; t < TL; ++t) {
    const int x = X0 + 16 * t + li;
    double chi = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int y = Y0 + 16 * wave + 4 * lg + j;
      if (x < c.nx && y < c.ny) {
        const size_t p = size_t(y) * c.nx + x;
        const float m = float(dacc[t][j] * unscale);
        if (out) AT(out, size_t(img) * c.nx * c.ny + p) = m;
        if (partial) chi += chi2_pixel<float>(c, p, m, img);
        if (c.gout)
          AT(static_cast<float *>(c.gout), size_t(img) * c.nx * c.ny + p) = float(dlogl_dm(c, p, double(m), img));
      }
    }
    if (partial) {
      for (int off = 32; off > 0; off >>= 1) chi += __shfl_xor(chi, off, 64);
      const int tx16 = (X0 >> 4) + t;
      // tiles past the image's edge hold no pixel and have no slot
      if (lane == 0 && 16 * tx16 < c.nx && 16 * ty16 < c.ny)
        AT(partial, size_t(img) * n16 + size_t(ty16) * n16x + tx16) = chi;
    }
  }
}

// ------------------------------------------------------------- gradient ---
// Number of kwargs of a profile type (its slots in a parameter block).
__host__ __device__ constexpr int n_params_of(int type) {
  switch (type) {
    case LENSIM_EPL: return 6;
    case LENSIM_SIE: return 5;
    case LENSIM_NIE: return 6;
    case LENSIM_NFW: return 4;
    case LENSIM_TNFW: return 5;
    case LENSIM_SHEAR: return 4;
    case LENSIM_CONVERGENCE: return 3;
    case LENSIM_SERSIC: return 5;
    case LENSIM_SERSIC_ELLIPSE: return 7;
    case LENSIM_GAUSSIAN: return 4;
    default: return 0;
  }
}

struct GradArgs {
  const double *params;   // [n_img][n_prof][8]
  const double *coefd;    // EPL F_n (double)
  const float *coeff;     // EPL F_n (float)
  const double *dcoefd;   // EPL dF_n/dt
  const float *dcoeff;
  const void *glow;       // [n_img][ny][nx] dlogL / d(unconvolved image), compute type
  double *gpart;          // [n_img][n_prof][nblk][8]
  void *gbeta;            // [n_img][ny][nx][s][s][2] dS/dbeta of the sources' sum, compute type, or NULL
  bool kept;              // gbeta holds beta (from the render) until the source's launch puts dS/dbeta there
  void *beta;             // same shape: beta (bulk and multi-plane lists, by the render or the adjoint kernels), or NULL
};

// A light profile's flux and its derivatives in its own kwargs (the N seeds
// of ps) at (x, y): closed form for SERSIC_ELLIPSE, duals otherwise.
template <typename T, int N>
__device__ __forceinline__ gm::Dual<T, N> light_grad(int type, const gm::Dual<T, N> *ps, const double *rd,
                                                     const double *pk, T x, T y) {
  using S = gm::Dual<T, N>;
  if constexpr (N == 7) {
    if (type == LENSIM_SERSIC_ELLIPSE) {
      T gp[7], gx, gy;
      S r;
      r.v = gm::sersic_ellipse_grad_rec<T>(rd, pk, x, y, gp, gx, gy);
#pragma unroll
      for (int i = 0; i < 7; ++i) r.d[i] = gp[i];
      return r;
    }
  }
  return gm::light_g<T, S>(type, ps, S(x), S(y));
}

// Sum of the source light profiles at beta and its gradient in beta (the
// tangents d[0], d[1]): closed form for SERSIC_ELLIPSE, two dual seeds
// otherwise.
template <typename T>
__device__ __forceinline__ gm::Dual<T, 2> sources_at(const ModelArgs &m, const GradArgs &ga, const RecPtrs<T> &rp,
                                                     int img, T bx, T by) {
  using S2 = gm::Dual<T, 2>;
  const S2 bx2 = S2::seed(bx, 0), by2 = S2::seed(by, 1);
  S2 f2 = S2(T(0));
  for (int j = m.n_defl; j < m.n_defl + m.n_source; ++j) {
    const double *pj = ga.params + (size_t(img) * m.n_prof + j) * LENSIM_NPARAM;
    CHECK_SPAN(pj, LENSIM_NPARAM * sizeof(double));
    const int tj = m.types[j - m.n_bulk];
    if (tj == LENSIM_SERSIC_ELLIPSE) {
      T gp[7], gx, gy;
      f2.v += gm::sersic_ellipse_grad_rec<T>(rp.recd + j * kRec, pj, bx, by, gp, gx, gy);
      f2.d[0] += gx;
      f2.d[1] += gy;
      continue;
    }
    S2 pl[LENSIM_NPARAM];
#pragma unroll
    for (int i = 0; i < LENSIM_NPARAM; ++i) pl[i] = S2(T(pj[i]));
    f2 = f2 + gm::light_g<T, S2>(tj, pl, bx2, by2);
  }
  return f2;
}

// Contribution of one ray to d flux / d(kwargs of profile k), with the
// profile's own kwargs as N dual seeds; w = dlogL / d(ray flux).
// gb: this ray's dS/dbeta of the sources' sum (two values), when the model
// has inline lenses and sources: the first source's launch writes it, the lens
// launches (which run after it) read it instead of deflecting by the other
// deflectors and evaluating the sources again.  bt: this ray's beta, where the
// render or an adjoint kernel stored it (and an adjoint kernel gb) before.
// A lens with a live ray always has gb.  The float forms of ray_grad and
// lens_ray_grad keep the branch without it all the same: with it gone the
// compiler contracts the arithmetic of the other one differently, and the mixed
// gradient moves by 2.7e-8 of itself.
template <typename T, int N, bool HALO>
__device__ __forceinline__ void ray_grad(const ModelArgs &m, const GradArgs &ga, const RecPtrs<T> &rp, int img,
                                         int k, int type, double x, double y, double w, double *acc, T *gb,
                                         const T *bt) {
  using S = gm::Dual<T, N>;
  const double *pk = ga.params + (size_t(img) * m.n_prof + k) * LENSIM_NPARAM;
  CHECK_SPAN(pk, LENSIM_NPARAM * sizeof(double));
  S ps[LENSIM_NPARAM];
#pragma unroll
  for (int i = 0; i < LENSIM_NPARAM; ++i) ps[i] = i < N ? S::seed(T(pk[i]), i) : S(T(pk[i]));
  S flux;
  if constexpr (sizeof(T) == sizeof(double)) __builtin_assume(k >= m.n_lens || gb);
  if (k < m.n_lens && gb) {
    // d flux = dS/dbeta . d beta, d beta = -alpha_scaling d alpha_k
    S ax = S(T(0)), ay = S(T(0));
    gm::defl_g<T, S>(type, ps, S(T(x)), S(T(y)), ax, ay);
    const T gx = AT(gb, 0), gy = AT(gb, 1), as = T(m.alpha_scaling);
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] += w * double(-as * (gx * ax.d[i] + gy * ay.d[i]));
    return;
  }
  if (k < m.n_lens) {
    // d/d(lens kwargs): the other deflectors in the forward form, this one in duals
    double axp = 0.0, ayp = 0.0;
    for (int j = 0; j < m.n_lens; ++j) {
      if (j == k) continue;
      const int e = m.epl_index[j];
      const size_t co = (e >= 0) ? (size_t(img) * m.n_epl + e) * LENSIM_EPL_NMAX : 0;
      add_deflection<T, HALO>(m.types[j], Rec<T>{rp.recd + j * kRec, rp.rect + j * kRec}, rp.coefd + co,
                              rp.coeft + co, x, y, axp, ayp);
    }
    deflect_bulk<T, HALO>(m, rp, x, y, axp, ayp);
    S ax = S(T(axp)), ay = S(T(ayp));
    const S xs = S(T(x)), ys = S(T(y));
    gm::defl_g<T, S>(type, ps, xs, ys, ax, ay);
    const S bx = xs - ax * T(m.alpha_scaling), by = ys - ay * T(m.alpha_scaling);
    // the sources' gradient in beta, chained into this deflector's kwargs:
    // d flux = dS/dbeta_x d beta_x + dS/dbeta_y d beta_y
    const gm::Dual<T, 2> f2 = sources_at<T>(m, ga, rp, img, bx.v, by.v);
    flux.v = f2.v;
#pragma unroll
    for (int i = 0; i < N; ++i) flux.d[i] = f2.d[0] * bx.d[i] + f2.d[1] * by.d[i];
  } else if (k < m.n_defl + m.n_source) {
    // d/d(source kwargs) at the deflected position
    T bxs, bys;
    if (bt) {
      bxs = AT(bt, 0);
      bys = AT(bt, 1);
    } else {
      double ax = 0.0, ay = 0.0;
      deflect_all<T, HALO>(m, rp, img, x, y, ax, ay);
      bxs = T(x - ax * m.alpha_scaling);
      bys = T(y - ay * m.alpha_scaling);
    }
    bool done = false;
    if (gb && !bt) {  // the first source's launch: also dS/dbeta of the sources' sum for the lens launches
      if constexpr (N == 7) {
        if (m.n_source == 1 && type == LENSIM_SERSIC_ELLIPSE) {  // one evaluation gives both
          T gp[7], gx, gy;
          flux.v = gm::sersic_ellipse_grad_rec<T>(rp.recd + k * kRec, pk, bxs, bys, gp, gx, gy);
#pragma unroll
          for (int i = 0; i < 7; ++i) flux.d[i] = gp[i];
          AT(gb, 0) = gx;
          AT(gb, 1) = gy;
          done = true;
        }
      }
      if (!done) {
        const gm::Dual<T, 2> f2 = sources_at<T>(m, ga, rp, img, bxs, bys);
        AT(gb, 0) = f2.d[0];
        AT(gb, 1) = f2.d[1];
      }
    }
    if (!done) flux = light_grad<T, N>(type, ps, rp.recd + k * kRec, pk, bxs, bys);
  } else {
    // d/d(lens light kwargs) at the ray
    flux = light_grad<T, N>(type, ps, rp.recd + k * kRec, pk, T(x), T(y));
  }
#pragma unroll
  for (int i = 0; i < N; ++i) acc[i] += w * double(flux.d[i]);
}

// ray_grad for an inline NFW deflector k, its closed forms in double in both
// forms (the NFW family's float ones cancel); gb: dS/dbeta.
template <typename T>
__device__ __forceinline__ void nfw_ray_grad(const ModelArgs &m, const GradArgs &ga, const RecPtrs<T> &rp, int img,
                                             int k, double x, double y, double w, double *acc, const T *gb) {
  const double *pk = ga.params + (size_t(img) * m.n_prof + k) * LENSIM_NPARAM;
  CHECK_SPAN(pk, LENSIM_NPARAM * sizeof(double));
  double a_x, a_y, dax[4], day[4];
  gm::nfw_dalpha_f64(rp.recd + k * kRec, pk, x, y, a_x, a_y, dax, day);
  const double gx = double(AT(gb, 0)), gy = double(AT(gb, 1)), as = m.alpha_scaling;
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] += w * (-as * (gx * dax[i] + gy * day[i]));
}

// The deflection of the EPL deflector k at (x, y) and its derivatives by the
// six kwargs (theta_E, gamma, e1, e2, center_x, center_y).  Two dual seeds
// carry gamma and the axis ratio q; the rest is in closed form:
//  * alpha scales as b^t with b = theta_E sqrt(q), so d alpha / d theta_E =
//    t alpha / theta_E;
//  * d alpha / d center = -H, H = d alpha / dx the Hessian, written as the
//    reference's EPLMajorAxis.hessian (LensModel/Profiles/epl.py:398-440, and
//    the rotation of :203-232): kappa = (2 - t)/2 (b/R)^t and the shear of
//    its eq. (17) from alpha itself;
//  * alpha(x) = R(phi) alpha_M(R(phi)^T (x - c)), so d alpha / d phi =
//    J alpha - H J (x - c) with J the quarter turn;
//  * (e1, e2) -> (phi, q) by the closed forms of Util/param_util.py:88-100
//    (phi = atan2(e2, e1) / 2, c = min(|e|, 0.9999), q = (1 - c) / (1 + c);
//    dq = 0 where c is clamped).
template <typename T>
__device__ __forceinline__ void epl_dalpha(const ModelArgs &m, const GradArgs &ga, const RecPtrs<T> &rp, int img,
                                           int k, const double *pk, double x, double y, T &a_x, T &a_y, T *dax,
                                           T *day) {
  if constexpr (sizeof(T) == sizeof(double)) {
    const size_t co = (size_t(img) * m.n_epl + m.epl_index[k]) * LENSIM_EPL_NMAX;
    CHECK_SPAN(ga.coefd + co, LENSIM_EPL_NMAX * sizeof(double));
    CHECK_SPAN(ga.dcoefd + co, LENSIM_EPL_NMAX * sizeof(double));
    gm::epl_dalpha_f64(rp.recd + k * kRec, ga.coefd + co, ga.dcoefd + co, pk, x, y, a_x, a_y, dax, day);
    return;
  }
  using S = gm::Dual<T, 2>;
  S ps[LENSIM_NPARAM];
#pragma unroll
  for (int i = 0; i < LENSIM_NPARAM; ++i) ps[i] = i == 1 ? S::seed(T(pk[1]), 0) : S(T(pk[i]));
  const int e = m.epl_index[k];
  const size_t co = (size_t(img) * m.n_epl + e) * LENSIM_EPL_NMAX;
  const int nser = int(rp.recd[k * kRec + EPL_NF]);  // the float form
  const T *c = reinterpret_cast<const T *>(ga.coeff + co), *dc = reinterpret_cast<const T *>(ga.dcoeff + co);
  CHECK_SPAN(c, LENSIM_EPL_NMAX * sizeof(T));
  CHECK_SPAN(dc, LENSIM_EPL_NMAX * sizeof(T));
  // q, cos phi and sin phi from the record, not per ray
  const double *rdk = rp.recd + k * kRec;
  const T q = T(rdk[EPL_Q]), cs = T(rdk[EPL_C]), sn = T(rdk[EPL_S]);
  S ax = S(T(0)), ay = S(T(0));
  gm::epl_g_geo<T>(ps, S::seed(q, 1), S(cs), S(sn), c, dc, nser, S(T(x)), S(T(y)), ax, ay);
  a_x = ax.v;
  a_y = ay.v;
  const T thetaE = T(pk[0]), t = T(pk[1]) - T(1);
  const T dth = thetaE != T(0) ? t / thetaE : T(0);
  dax[0] = a_x * dth;
  day[0] = a_y * dth;
  dax[1] = ax.d[0];
  day[1] = ay.d[0];
  // Hessian in the major-axis frame, rotated back
  const T dx = T(x) - T(pk[4]), dy = T(y) - T(pk[5]);
  const T xr = dx * cs + dy * sn, yr = dy * cs - dx * sn;
  const T r = gm::sqrt(xr * xr + yr * yr);
  T fxx = T(0), fxy = T(0), fyy = T(0);
  if (r > T(0)) {
    T R = gm::sqrt(q * q * xr * xr + yr * yr);
    R = R >= T(0.00000001) ? R : T(0.00000001);
    const T kappa = (T(2) - t) / T(2) * gm::exp(t * (T(rdk[EPL_LNB]) - gm::log(R)));  // (b/R)^t
    const T ct = xr / r, st = yr / r;
    const T c2 = ct * ct * T(2) - T(1), s2 = st * ct * T(2);
    const T fr = a_x * cs + a_y * sn, fi = a_y * cs - a_x * sn;  // alpha in the major-axis frame
    const T g1 = (T(1) - t) * (fr * ct - fi * st) / r - kappa * c2;
    const T g2 = (T(1) - t) * (fi * ct + fr * st) / r - kappa * s2;
    const T c2p = cs * cs - sn * sn, s2p = T(2) * sn * cs;
    const T G1 = c2p * g1 - s2p * g2, G2 = s2p * g1 + c2p * g2;
    fxx = kappa + G1;
    fyy = kappa - G1;
    fxy = G2;
  }
  // orientation: d alpha / d phi = J alpha - H J (x - c)
  const T dphx = fxx * dy - fxy * dx - a_y, dphy = fxy * dy - fyy * dx + a_x;
  const T e1 = T(pk[2]), e2 = T(pk[3]);
  const T c2 = e1 * e1 + e2 * e2, ce = gm::sqrt(c2);
  const T h = T(0.5) / c2;  // d phi / d(e1, e2) = (-e2, e1) / (2 c^2)
  const T dp1 = -e2 * h, dp2 = e1 * h;
  const T dqdc = ce < T(0.9999) ? T(-2) / ((T(1) + ce) * (T(1) + ce)) : T(0);
  const T dq1 = dqdc * e1 / ce, dq2 = dqdc * e2 / ce;
  dax[2] = ax.d[1] * dq1 + dphx * dp1;
  day[2] = ay.d[1] * dq1 + dphy * dp1;
  dax[3] = ax.d[1] * dq2 + dphx * dp2;
  day[3] = ay.d[1] * dq2 + dphy * dp2;
  dax[4] = -fxx;
  day[4] = -fxy;
  dax[5] = -fxy;
  day[5] = -fyy;
}

// The deflection of the SIE / NIE deflector k at (x, y) and its derivatives by
// its kwargs (theta_E, e1, e2[, s_scale], center_x, center_y).  Dual seeds
// carry q, s_scale and the centre; the axis ratio and orientation come from
// the ellipticity (q, by Util/param_util.py:88-100) and the record (cos phi,
// sin phi), not per-ray dual atan2 / cos / sin; alpha is linear in theta_E
// (b = theta_E sqrt(q)); d alpha / d phi = J alpha - H J (x - c) as for the
// EPL, H = -(d alpha / d center).
template <typename T, int TYPE>
__device__ __forceinline__ void nie_dalpha(const double *rd, const double *pk, double x, double y, T &a_x, T &a_y,
                                           T *dax, T *day) {
  if constexpr (sizeof(T) == sizeof(double)) {
    gm::nie_dalpha_f64<TYPE>(rd, pk, x, y, a_x, a_y, dax, day);
    return;
  }
  using S = gm::Dual<T, 4>;  // q, s_scale, center_x, center_y
  constexpr bool kNie = TYPE == LENSIM_NIE;
  const T e1 = T(pk[1]), e2 = T(pk[2]);
  const T c2 = e1 * e1 + e2 * e2, ce = gm::sqrt(c2);
  const T cc = ce < T(0.9999) ? ce : T(0.9999);
  const T q = (T(1) - cc) / (T(1) + cc);
  const T s_scale = kNie ? T(pk[3]) : T(0.0000000001);
  const T cx = T(pk[kNie ? 4 : 3]), cy = T(pk[kNie ? 5 : 4]);
  S ax = S(T(0)), ay = S(T(0));
  gm::nie_g_geo<T>(S(T(pk[0])), S::seed(q, 0), S(T(rd[NIE_C])), S(T(rd[NIE_S])), S::seed(s_scale, 1),
                   S::seed(cx, 2), S::seed(cy, 3), S(T(x)), S(T(y)), ax, ay);
  a_x = ax.v;
  a_y = ay.v;
  const T thetaE = T(pk[0]);
  const T ith = thetaE != T(0) ? T(1) / thetaE : T(0);
  dax[0] = a_x * ith;
  day[0] = a_y * ith;
  // H = d alpha / d(x, y) = -(d alpha / d center)
  const T hxx = -ax.d[2], hxy = -ax.d[3], hyx = -ay.d[2], hyy = -ay.d[3];
  const T dx = T(x) - cx, dy = T(y) - cy;
  const T dphx = hxx * dy - hxy * dx - a_y, dphy = hyx * dy - hyy * dx + a_x;
  const T h = T(0.5) / c2;  // d phi / d(e1, e2) = (-e2, e1) / (2 c^2)
  const T dp1 = -e2 * h, dp2 = e1 * h;
  const T dqdc = ce < T(0.9999) ? T(-2) / ((T(1) + ce) * (T(1) + ce)) : T(0);
  const T dq1 = dqdc * e1 / ce, dq2 = dqdc * e2 / ce;
  dax[1] = ax.d[0] * dq1 + dphx * dp1;
  day[1] = ay.d[0] * dq1 + dphy * dp1;
  dax[2] = ax.d[0] * dq2 + dphx * dp2;
  day[2] = ay.d[0] * dq2 + dphy * dp2;
  constexpr int kc = kNie ? 4 : 3;  // the centre's slots
  if constexpr (kNie) {
    dax[3] = ax.d[1];
    day[3] = ay.d[1];
  }
  dax[kc] = ax.d[2];
  day[kc] = ay.d[2];
  dax[kc + 1] = ax.d[3];
  day[kc + 1] = ay.d[3];
}

// Contribution of one ray to d flux / d(kwargs of the EPL, SIE or NIE deflector k).
template <typename T, bool HALO, int TYPE = LENSIM_EPL>
__device__ __forceinline__ void lens_ray_grad(const ModelArgs &m, const GradArgs &ga, const RecPtrs<T> &rp, int img,
                                             int k, double x, double y, double w, double *acc, const T *gb) {
  const double *pk = ga.params + (size_t(img) * m.n_prof + k) * LENSIM_NPARAM;
  CHECK_SPAN(pk, LENSIM_NPARAM * sizeof(double));
  double axp = 0.0, ayp = 0.0;  // the other deflectors in the forward form (not needed with gb)
  if (!gb) {
    for (int j = 0; j < m.n_lens; ++j) {
      if (j == k) continue;
      const int ej = m.epl_index[j];
      const size_t coj = (ej >= 0) ? (size_t(img) * m.n_epl + ej) * LENSIM_EPL_NMAX : 0;
      add_deflection<T, HALO>(m.types[j], Rec<T>{rp.recd + j * kRec, rp.rect + j * kRec}, rp.coefd + coj,
                              rp.coeft + coj, x, y, axp, ayp);
    }
    deflect_bulk<T, HALO>(m, rp, x, y, axp, ayp);
  }
  T a_x, a_y, dax[6], day[6];
  if constexpr (TYPE == LENSIM_EPL)
    epl_dalpha<T>(m, ga, rp, img, k, pk, x, y, a_x, a_y, dax, day);
  else
    nie_dalpha<T, TYPE>(rp.recd + k * kRec, pk, x, y, a_x, a_y, dax, day);
  constexpr int N = n_params_of(TYPE);
  const T as = T(m.alpha_scaling);
  T gx, gy;
  if (gb) {
    gx = AT(gb, 0);
    gy = AT(gb, 1);
  } else {
    const T bxv = T(x) - (T(axp) + a_x) * as, byv = T(y) - (T(ayp) + a_y) * as;
    const gm::Dual<T, 2> f2 = sources_at<T>(m, ga, rp, img, bxv, byv);
    gx = f2.d[0];
    gy = f2.d[1];
  }
#pragma unroll
  for (int i = 0; i < N; ++i) acc[i] += w * double(-as * (gx * dax[i] + gy * day[i]));
}

// One block = kGradPix x 256 pixels x one image of profile k, whose type
// TYPE is fixed at compile time (one launch per profile: each type's kernel
// keeps only its own registers and code); each thread takes kGradPix pixels
// 256 apart, so the block reduction and the per-thread set-up are shared by
// kGradPix pixels' rays.
// The float form is held to 128 VGPRs (four waves per SIMD instead of three
// for the EPL's duals; no spills): 239k -> 250k gradients/s.  The FP64 form,
// and the double closed forms of NFW / TNFW, would spill.  What bounds it in
// FP64 is the vector unit's instructions: the closed forms of grad.hpp in place
// of duals took 64 images of 120^2 (EPL + SHEAR, Sersic source and light) from
// 620 to 411 us a call, sums of their bases with the kwargs' factors applied
// once a block (a square root and five divisions a ray less) from 391 to 351,
// and the source's rays taken from the render (MpKeep, GradArgs::kept) to 309.
template <typename T, int TYPE>
constexpr int grad_waves_per_eu() {
  return (sizeof(T) == sizeof(float) && TYPE != LENSIM_NFW && TYPE != LENSIM_TNFW) ? 4 : 1;
}

template <typename T, bool HALO, int TYPE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(grad_waves_per_eu<T, TYPE>()))) void
grad_kernel(ModelArgs m, GridArgs g, GradArgs ga,
                                                   const double *__restrict__ recd, const float *__restrict__ recf,
                                                   const double *__restrict__ coefd, const float *__restrict__ coeff,
                                                   int k) {
  const int img = blockIdx.y;
  const int npix = g.nx * g.ny;
  const RecPtrs<T> rp = rec_ptrs<T>(m, recd, recf, coefd, coeff, img);
  constexpr int type = TYPE;
  T *gbeta = static_cast<T *>(ga.gbeta);
  double acc[LENSIM_NPARAM];
#pragma unroll
  for (int q = 0; q < LENSIM_NPARAM; ++q) acc[q] = 0.0;
  // FP64: sums of the closed forms' bases, whose factors of the kwargs alone are applied below
  constexpr bool kF64 = sizeof(T) == sizeof(double);
  constexpr bool kEll = kF64 && (type == LENSIM_EPL || type == LENSIM_SIE || type == LENSIM_NIE);
  constexpr bool kSersic = kF64 && type == LENSIM_SERSIC_ELLIPSE;
  const double *rd = rp.recd + k * kRec, *pk = ga.params + (size_t(img) * m.n_prof + k) * LENSIM_NPARAM;
  CHECK_SPAN(pk, LENSIM_NPARAM * sizeof(double));
  const gm::EllKw ek = kEll ? gm::EllKw(pk[type == LENSIM_EPL ? 2 : 1], pk[type == LENSIM_EPL ? 3 : 2]) : gm::EllKw();
  std::conditional_t<kSersic, gm::SersicGrad, const double *> sersic(rd);
  bool seen = false;  // whether the thread has a ray: without one its sums are 0 whatever the kwargs' factors are
  for (int pp = 0; pp < kGradPix; ++pp) {
  const int pix0 = (blockIdx.x * kGradPix + pp) * blockDim.x + threadIdx.x;
  const bool active = pix0 < npix;
  const int pix = active ? pix0 : npix - 1;
  int i;
  const int j = div_by(pix, g.nx, g.inv_nx, i);
  // the pixel's flux is scale * flux_scaling * (sum over its rays)
  const double w = active ? double(AT(static_cast<const T *>(ga.glow), size_t(img) * npix + pix)) * g.scale *
                                m.flux_scaling
                          : 0.0;
  const double ra_c = i * g.m00 + j * g.m01 + g.ra0;
  const double dec_c = i * g.m10 + j * g.m11 + g.dec0;
  const double inv_s = g.inv_s;
  const double o0 = g.o0;
  // a lens profile only matters if a source is there to be lensed
  const bool live = active && w != 0.0 && (k >= m.n_defl || m.n_source > 0) && evaluated(g, i, j);
  seen |= live;
  for (int sy = 0; live && sy < g.s; ++sy) {
    const double oy = o0 + sy * inv_s;
    for (int sx = 0; sx < g.s; ++sx) {
      const double ox = o0 + sx * inv_s;
      const double x = ra_c + g.m00 * ox + g.m01 * oy;
      const double y = dec_c + g.m10 * ox + g.m11 * oy;
      // this ray's slots: dS/dbeta, written by the first source's launch (or an adjoint kernel) and read by
      // the inline lens launches; beta, written by the render or an adjoint kernel and read by the source launches
      const size_t slot = ((size_t(img) * npix + pix) * size_t(g.s * g.s) + size_t(sy * g.s + sx)) * 2;
      T *gb = (gbeta && (k < m.n_lens || k == m.n_defl)) ? gbeta + slot : nullptr;
      const T *bt = (ga.beta && k >= m.n_defl && k < m.n_defl + m.n_source) ? static_cast<const T *>(ga.beta) + slot
                                                                            : nullptr;
      if (gb) CHECK_SPAN(gb, 2 * sizeof(T));
      if (bt) CHECK_SPAN(bt, 2 * sizeof(T));
      if constexpr (kEll) {
        double bx[6], by[6];
        const double lw = -m.alpha_scaling * w, lx = lw * double(AT(gb, 0)), ly = lw * double(AT(gb, 1));
        if constexpr (type == LENSIM_EPL) {
          const size_t co = (size_t(img) * m.n_epl + m.epl_index[k]) * LENSIM_EPL_NMAX;
          CHECK_SPAN(ga.coefd + co, LENSIM_EPL_NMAX * sizeof(double));
          CHECK_SPAN(ga.dcoefd + co, LENSIM_EPL_NMAX * sizeof(double));
          gm::epl_basis_f64(rd, ga.coefd + co, ga.dcoefd + co, x, y, bx, by);
        } else {
          gm::nie_basis_f64<type>(rd, ek.q0, x, y, bx, by);
        }
#pragma unroll
        for (int q = 0; q < n_params_of(type); ++q) acc[q] += fma(lx, bx[q], ly * by[q]);
      } else if constexpr (kSersic) {
        double px = x, py = y, gx, gy;
        if (k < m.n_defl + m.n_source) {
          if (bt) {
            px = double(AT(bt, 0));
            py = double(AT(bt, 1));
          } else if (ga.kept) {
            px = double(AT(gb, 0));
            py = double(AT(gb, 1));
          } else {
            trace_ray<T, HALO, false>(m, rp, img, x, y, px, py);
          }
        }
        sersic.add(px, py, w, gx, gy);
        if (gb && !bt) {  // the first source's launch, for the lens launches
          if (m.n_source > 1) {
            const gm::Dual<T, 2> f2 = sources_at<T>(m, ga, rp, img, T(px), T(py));
            gx = double(f2.d[0]);
            gy = double(f2.d[1]);
          }
          AT(gb, 0) = T(gx);
          AT(gb, 1) = T(gy);
        }
      }
      else if constexpr (type == LENSIM_EPL) lens_ray_grad<T, HALO>(m, ga, rp, img, k, x, y, w, acc, gb);
      else if constexpr (type == LENSIM_SIE) lens_ray_grad<T, HALO, LENSIM_SIE>(m, ga, rp, img, k, x, y, w, acc, gb);
      else if constexpr (type == LENSIM_NIE) lens_ray_grad<T, HALO, LENSIM_NIE>(m, ga, rp, img, k, x, y, w, acc, gb);
      else if constexpr (type == LENSIM_NFW) nfw_ray_grad<T>(m, ga, rp, img, k, x, y, w, acc, gb);
      else if constexpr (type == LENSIM_TNFW) {  // live and a lens: gb is there
        const double lw = -m.alpha_scaling * w;
        tnfw_ray_grad(TnfwRec(rp.recd + k * kRec), rp.recd + k * kRec, x, y, lw * double(AT(gb, 0)),
                      lw * double(AT(gb, 1)), acc);
      }
      else if constexpr (type == LENSIM_SHEAR) ray_grad<T, 4, HALO>(m, ga, rp, img, k, type, x, y, w, acc, gb, bt);
      else if constexpr (type == LENSIM_CONVERGENCE)
        ray_grad<T, 3, HALO>(m, ga, rp, img, k, type, x, y, w, acc, gb, bt);
      else if constexpr (type == LENSIM_SERSIC) ray_grad<T, 5, HALO>(m, ga, rp, img, k, type, x, y, w, acc, gb, bt);
      else if constexpr (type == LENSIM_SERSIC_ELLIPSE)
        ray_grad<T, 7, HALO>(m, ga, rp, img, k, type, x, y, w, acc, gb, bt);
      else if constexpr (type == LENSIM_GAUSSIAN) ray_grad<T, 4, HALO>(m, ga, rp, img, k, type, x, y, w, acc, gb, bt);
    }
  }
  }
  if (seen) {
    if constexpr (type == LENSIM_TNFW) tnfw_grad_scale(rd, acc);
    if constexpr (kEll && type == LENSIM_EPL) gm::epl_kw(ek, rd, pk, acc);
    if constexpr (kEll && type != LENSIM_EPL) gm::nie_kw<type>(ek, pk, acc);
    if constexpr (kSersic) sersic.kwargs(rd, pk, acc);
  }
  // block sum of the 8 accumulators in a fixed order
  __shared__ double red[256 / 64][LENSIM_NPARAM];
#pragma unroll
  for (int q = 0; q < LENSIM_NPARAM; ++q) {
    double v = acc[q];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][q] = v;
  }
  __syncthreads();
  if (threadIdx.x < LENSIM_NPARAM) {
    double v = 0.0;
    for (int wv = 0; wv < int(blockDim.x >> 6); ++wv) v += red[wv][threadIdx.x];
    AT(ga.gpart, ((size_t(img) * m.n_prof + k) * gridDim.x + blockIdx.x) * LENSIM_NPARAM + threadIdx.x) = v;
  }
}

// grad_kernel for profile k of the model (its type read on the host).
template <typename T, bool HALO>
int launch_grad_profile(const ModelArgs &m, const GridArgs &g, const GradArgs &ga, const double *recd,
                        const float *recf, int nblk, int n_img, int k, hipStream_t st) {
  const dim3 grid(nblk, n_img);
#define LENSIM_GRAD(TY)                                                                                     \
  grad_kernel<T, HALO, TY><<<grid, 256, 0, st>>>(m, g, ga, recd, recf, ga.coefd, ga.coeff, k)
  switch (type_of(m, k)) {
    case LENSIM_EPL: LENSIM_GRAD(LENSIM_EPL); break;
    case LENSIM_SIE: LENSIM_GRAD(LENSIM_SIE); break;
    case LENSIM_NIE: LENSIM_GRAD(LENSIM_NIE); break;
    case LENSIM_NFW:  // present only in a model with halos (HALO)
      if constexpr (HALO) LENSIM_GRAD(LENSIM_NFW); else LENSIM_GRAD(LENSIM_NULL);
      break;
    case LENSIM_TNFW:
      if constexpr (HALO) LENSIM_GRAD(LENSIM_TNFW); else LENSIM_GRAD(LENSIM_NULL);
      break;
    case LENSIM_SHEAR: LENSIM_GRAD(LENSIM_SHEAR); break;
    case LENSIM_CONVERGENCE: LENSIM_GRAD(LENSIM_CONVERGENCE); break;
    case LENSIM_SERSIC: LENSIM_GRAD(LENSIM_SERSIC); break;
    case LENSIM_SERSIC_ELLIPSE: LENSIM_GRAD(LENSIM_SERSIC_ELLIPSE); break;
    case LENSIM_GAUSSIAN: LENSIM_GRAD(LENSIM_GAUSSIAN); break;
    default: LENSIM_GRAD(LENSIM_NULL); break;  // no kwargs: the kernel writes zero partials
  }
#undef LENSIM_GRAD
  return check_launch("grad_kernel");
}

// Deflector k's deflection at (x, y) and its derivatives by its kwargs,
// slots 0 .. N-1: the EPL's in the compute type, the other types' closed forms
// in double.  The last two slots of every deflector type are its centre, whose
// derivative is minus the column of d alpha / d(x, y).
// N = n_params_of(TYPE) derivatives of a closed form, laid out for deflector_dalpha.
template <int N>
__device__ __forceinline__ void spread_dalpha(const double *dx, const double *dy, double *dax, double *day,
                                              double *dcen) {
#pragma unroll
  for (int i = 0; i < LENSIM_NPARAM; ++i) {
    dax[i] = i < N ? dx[i] : 0.0;
    day[i] = i < N ? dy[i] : 0.0;
  }
  dcen[0] = dx[N - 2];
  dcen[1] = dy[N - 2];
  dcen[2] = dx[N - 1];
  dcen[3] = dy[N - 1];
}

template <typename T, bool HALO>
__device__ __forceinline__ void deflector_dalpha(const ModelArgs &m, const GradArgs &ga, const RecPtrs<T> &rp,
                                                 int img, int k, int type, double x, double y, double &ax,
                                                 double &ay, double *dax, double *day, double *dcen) {
  const double *pk = ga.params + (size_t(img) * m.n_prof + k) * LENSIM_NPARAM;
  CHECK_SPAN(pk, LENSIM_NPARAM * sizeof(double));
  switch (type) {
    case LENSIM_EPL: {
      T a_x, a_y, dx[6], dy[6];
      epl_dalpha<T>(m, ga, rp, img, k, pk, x, y, a_x, a_y, dx, dy);
      ax = double(a_x);
      ay = double(a_y);
#pragma unroll
      for (int i = 0; i < LENSIM_NPARAM; ++i) {
        dax[i] = i < 6 ? double(dx[i]) : 0.0;
        day[i] = i < 6 ? double(dy[i]) : 0.0;
      }
      dcen[0] = dax[4];
      dcen[1] = day[4];
      dcen[2] = dax[5];
      dcen[3] = day[5];
      break;
    }
    case LENSIM_SIE: {
      double dx[6], dy[6];
      nie_dalpha<double, LENSIM_SIE>(rp.recd + k * kRec, pk, x, y, ax, ay, dx, dy);
      spread_dalpha<5>(dx, dy, dax, day, dcen);
      break;
    }
    case LENSIM_NIE: {
      double dx[6], dy[6];
      nie_dalpha<double, LENSIM_NIE>(rp.recd + k * kRec, pk, x, y, ax, ay, dx, dy);
      spread_dalpha<6>(dx, dy, dax, day, dcen);
      break;
    }
    case LENSIM_NFW:
      if constexpr (HALO) {
        double dx[4], dy[4];
        gm::nfw_dalpha_f64(rp.recd + k * kRec, pk, x, y, ax, ay, dx, dy);
        spread_dalpha<4>(dx, dy, dax, day, dcen);
      }
      break;
    default: break;  // TNFW, SHEAR and CONVERGENCE: their callers' closed forms
  }
}

// ---- gradient of bulk and multi-plane deflector lists ----
// d flux / d(kwargs) of every deflector takes two steps.  An adjoint kernel
// traces each ray and stores, per run of deflectors on one plane (one run for
// a single-plane list), the ray's position (x, y) and the adjoint (lx, ly) of
// the deflection there; then defl_grad_kernel sums lambda . d alpha_k /
// d kwargs_k over the rays, deflector by deflector.  So the serial part (the
// planes) holds no parameter sums, and those are taken with a lane per ray, in
// registers, with one wave sum per deflector at the end.  (One kernel that did
// both summed five parameters over each block at every deflector: 23.5 ms for
// 5256 deflectors and 100^2 rays, where the two steps take 0.50 and 0.26 ms.)

// Ray `first` + lane of image img (first + lane < the rays of the image, which
// may be more than 2^31 in a list on one plane): its index on the grid,
// position and the weight w = dlogL / d(ray flux); live: whether it has a weight
// and a source to hit.
struct GradRay {
  size_t slot;
  double x, y, w;
  bool live;
};
template <typename T>
__device__ __forceinline__ GradRay grad_ray(const ModelArgs &m, const GridArgs &g, const GradArgs &ga, int img,
                                            int64_t first, int lane, bool active) {
  const int npix = g.nx * g.ny, ss = g.s * g.s;
  int left, sub, i, sx;
  const int pix0 = int(div_by64(first, ss, g.inv_ss, left));
  const int pix = pix0 + div_by(left + lane, ss, g.inv_ss, sub);
  const int j = div_by(pix, g.nx, g.inv_nx, i), sy = div_by(sub, g.s, g.inv_s, sx);
  const double ox = g.o0 + sx * g.inv_s, oy = g.o0 + sy * g.inv_s;
  GradRay r;
  r.x = i * g.m00 + j * g.m01 + g.ra0 + g.m00 * ox + g.m01 * oy;
  r.y = i * g.m10 + j * g.m11 + g.dec0 + g.m10 * ox + g.m11 * oy;
  r.w = active ? double(AT(static_cast<const T *>(ga.glow), size_t(img) * npix + pix)) * g.scale * m.flux_scaling : 0.0;
  r.live = r.w != 0.0 && m.n_source > 0 && evaluated(g, i, j);
  r.slot = ((size_t(img) * npix + pix) * size_t(ss) + size_t(sub)) * 2;
  return r;
}

// (d alpha_k / dx)^T l of one deflector added to (jx, jy).
template <typename T, bool HALO, bool SUB>
__device__ __forceinline__ void adjoint_one(const ModelArgs &m, const GradArgs &ga, const RecPtrs<T> &rp, int img,
                                            int k, int type, double x, double y, double lx, double ly, double &jx,
                                            double &jy) {
  const double *rd = rp.recd + k * kRec;
  switch (type) {
    case LENSIM_TNFW:
      if constexpr (HALO) tnfw_adjoint(TnfwRec(rd), rd, x, y, lx, ly, jx, jy);
      break;
    case LENSIM_CONVERGENCE:
      jx = fma(rd[CV_KAPPA], lx, jx);
      jy = fma(rd[CV_KAPPA], ly, jy);
      break;
    case LENSIM_SHEAR:
      jx += rd[SH_G1] * lx + rd[SH_G2] * ly;
      jy += rd[SH_G2] * lx - rd[SH_G1] * ly;
      break;
    case LENSIM_NULL:
      break;
    default:
      if constexpr (!SUB) {
        double ax = 0.0, ay = 0.0, dax[LENSIM_NPARAM], day[LENSIM_NPARAM], dcen[4] = {0.0, 0.0, 0.0, 0.0};
        deflector_dalpha<T, HALO>(m, ga, rp, img, k, type, x, y, ax, ay, dax, day, dcen);
        jx -= lx * dcen[0] + ly * dcen[1];
        jy -= lx * dcen[2] + ly * dcen[3];
      }
      break;
  }
}

// The adjoint of the multi-plane recursion (MultiPlaneBulk.ray_shooting,
// LensModel/MultiPlane/multi_plane_bulk.py:152-212)
//   P_p = P_{p-1} + T_p A_{p-1},  A_p = A_{p-1} - f_p alpha_p(P_p / Tz_p),
//   beta = P_n / Tz_n  (P_{-1} = 0, A_{-1} = the ray's angle):
// from gP = w dS/dbeta / Tz_n and gA = 0 at the source plane backwards,
//   lambda_p = -f_p gA  (the adjoint of alpha_p),
//   gP += (d alpha_p / dx)^T lambda_p / Tz_p,  then gA += T_p gP.
// Forwards nothing is left to do where the render kept its rays (MpKeep); when
// they take more than a round, block_trace again, storing each run's position.
// Backwards the same split of a run's deflectors over the block's waves (they
// share position and lambda: gA does not change where T is 0).  Each ray's beta
// is stored too, for the source profiles' launches.  Bound by the runs' serial chain at few rays
// (a barrier and the deflectors' records per run), by the vector ALU at many.
template <typename T, bool HALO, bool SUB, bool SOLO>
__global__ __launch_bounds__(mp_threads_most(SUB, SOLO)) void mp_adjoint_kernel(
    ModelArgs m, GridArgs g, GradArgs ga, const double *__restrict__ recd, const float *__restrict__ recf,
    const double *__restrict__ coefd, const float *__restrict__ coeff, const int *__restrict__ tab_all, bool both,
    double4 *store, size_t per_img, int img0, int round, bool keeps, const double *__restrict__ all_tij,
    const double *__restrict__ all_tz, const double *__restrict__ all_r2p) {
  __shared__ MpRed<SOLO> red;
  const int img = img0 + blockIdx.y, lane = threadIdx.x & 63;
  const MpTab tab = mp_tab(m, tab_all, img);
  if (both && bool(tab.sub) != SUB) return;  // the other instantiation's launch takes it
  const int64_t r_all = int64_t(g.nx) * g.ny * g.s * g.s;
  const MpWave<SOLO> w(mp_classes(m.n_defl, r_all, SUB));
  const int64_t cap = round_rays(per_img, tab.n), in = int64_t(blockIdx.x) * 64;
  if (in >= cap || round * cap + in >= r_all) return;
  const int64_t first = round * cap + in;
  const bool active = first + lane < r_all;
  const RecPtrs<T> rp = rec_ptrs<T>(m, recd, recf, coefd, coeff, img);
  const GradRay ray = grad_ray<T>(m, g, ga, img, first, active ? lane : int(r_all - 1 - first), active);
  double4 *st = store + size_t(blockIdx.y) * per_img + in + lane;  // this ray's entry of run c at st[c * cap]
  if (!__any(ray.live)) {  // the same in every wave that holds the rays
    for (int c = SOLO ? 0 : w.wave; c < tab.n; c += SOLO ? 1 : w.nw) AT(st, c * cap) = double4{0.0, 0.0, 0.0, 0.0};
    return;
  }
  const size_t o = size_t(img) * size_t(m.mp_stride);
  const double *tij = all_tij + o, *tzs = all_tz + o, *r2p = all_r2p + o;
  T bx = T(0), by = T(0), *b = static_cast<T *>(ga.beta) + ray.slot;
  if (keeps && cap >= r_all) {  // the render kept the positions and beta (MpKeep)
    if (ray.live) {
      bx = AT(b, 0);
      by = AT(b, 1);
    }
  } else {
    double bxd, byd;
    block_trace<T, HALO, true, true, SUB, SOLO>(m, rp, tab, tij, tzs, r2p, img, ray.x, ray.y, w, red, bxd, byd,
                                          [&](int c, double x, double y) {
                                            if (w.lead()) AT(st, c * cap) = double4{x, y, 0.0, 0.0};
                                          });
    bx = T(bxd);
    by = T(byd);
    if (ray.live && w.lead()) {
      AT(b, 0) = bx;
      AT(b, 1) = by;
    }
  }
  if (tab.n == 0) return;
  const int nd = m.mp_n - 1;
  double gPx = 0.0, gPy = 0.0, gAx = 0.0, gAy = 0.0;
  if (ray.live) {
    const gm::Dual<T, 2> f2 = sources_at<T>(m, ga, rp, img, bx, by);
    const double tzn = AT(tzs, nd), dt = AT(tij, nd);
    gPx = ray.w * double(f2.d[0]) / tzn;
    gPy = ray.w * double(f2.d[1]) / tzn;
    gAx = dt * gPx;
    gAy = dt * gPy;
  }
  w.barrier();  // the positions are stored, the last sums read
  auto members = [&](int p0, int p1) { return p0 + lane < p1 ? AT(tab.who, p0 + lane) : 0; };
  int c = tab.n - 1, p0 = AT(tab.start, c), p1 = AT(tab.start, c + 1);
  int ks = members(p0, p1);
  double4 at = AT(st, c * cap);
  double dt = AT(tij, p0), itz = rcp_full(AT(tzs, p0)), f = AT(r2p, p0);
  for (; c >= 0; --c) {
    const int cn = c > 0 ? c - 1 : 0, q0 = AT(tab.start, cn);
    const int ks_next = members(q0, p0);
    const double4 at_next = AT(st, cn * cap);
    const double dt_next = AT(tij, q0), tz_next = AT(tzs, q0), f_next = AT(r2p, q0);
    const double lx = -f * gAx, ly = -f * gAy;
    double jx, jy;
    if (w.lead()) AT(st, c * cap) = double4{at.x, at.y, ray.live ? lx : 0.0, ray.live ? ly : 0.0};
    run_sum<SUB>(w, red, c & 1, p1 - p0, jx, jy, [&](int q, double &sx, double &sy) {
      const int k = __builtin_amdgcn_readlane(ks, q);
      adjoint_one<T, HALO, SUB>(m, ga, rp, img, k & ((1 << kWhoBits) - 1), k >> kWhoBits, at.x, at.y, lx, ly, sx, sy);
    });
    gPx = fma(jx, itz, gPx);
    gPy = fma(jy, itz, gPy);
    gAx = fma(dt, gPx, gAx);
    gAy = fma(dt, gPy, gAy);
    p1 = p0;
    p0 = q0;
    ks = ks_next;
    at = at_next;
    dt = dt_next;
    itz = rcp_full(tz_next);
    f = f_next;
  }
}

// The same for a single-plane list: with beta = theta - alpha_scaling sum_j
// alpha_j the adjoint of every deflection is l = -alpha_scaling w dS/dbeta.
// The block's waves share the bulk list of its 64 rays (the first takes the
// inline deflectors too); kept: the render kept beta, and the block is one
// wave.  Stores (x, y, l), beta, and dS/dbeta for the inline
// deflectors' launches.
constexpr int kBulkWaves = kSumWaves;
template <typename T, bool HALO>
__global__ __launch_bounds__(64 * kBulkWaves) void bulk_adjoint_kernel(
    ModelArgs m, GridArgs g, GradArgs ga, const double *__restrict__ recd, const float *__restrict__ recf,
    const double *__restrict__ coefd, const float *__restrict__ coeff, double4 *__restrict__ store, size_t per_img,
    int img0, int round, bool kept) {
  __shared__ WaveSums red;
  const int img = img0 + blockIdx.y, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t r_all = int64_t(g.nx) * g.ny * g.s * g.s;
  const int64_t cap = round_rays(per_img, 1), in = int64_t(blockIdx.x) * 64;
  if (in >= cap || round * cap + in >= r_all) return;
  const int64_t first = round * cap + in;
  const bool active = first + lane < r_all;
  const RecPtrs<T> rp = rec_ptrs<T>(m, recd, recf, coefd, coeff, img);
  const GradRay ray = grad_ray<T>(m, g, ga, img, first, active ? lane : int(r_all - 1 - first), active);
  double ax = 0.0, ay = 0.0;
  if (!kept && __any(ray.live)) {  // the same in every wave
    if (wave == 0)
      for (int k = 0; k < m.n_lens; ++k) deflect_one<T, HALO, false>(m, rp, img, k, m.types[k], ray.x, ray.y, ax, ay);
    for (int k = m.n_lens + wave; k < m.n_defl; k += kBulkWaves) {
      const int type = m.bulk_type ? m.bulk_type : AT(m.bulk_types, k - m.n_lens);
      deflect_one<T, HALO, false>(m, rp, img, k, type == LENSIM_EPL ? LENSIM_NULL : type, ray.x, ray.y, ax, ay);
    }
    across_waves(red, 0, kBulkWaves, ax, ay);
  }
  if (wave != 0) return;
  double lx = 0.0, ly = 0.0;
  if (ray.live) {
    const double as = m.alpha_scaling;
    T *b = static_cast<T *>(ga.beta) + ray.slot;
    const T bx = kept ? AT(b, 0) : T(ray.x - ax * as), by = kept ? AT(b, 1) : T(ray.y - ay * as);
    const gm::Dual<T, 2> f2 = sources_at<T>(m, ga, rp, img, bx, by);
    lx = -as * ray.w * double(f2.d[0]);
    ly = -as * ray.w * double(f2.d[1]);
    if (!kept) {
      AT(b, 0) = bx;
      AT(b, 1) = by;
    }
    if (ga.gbeta) {
      T *gb = static_cast<T *>(ga.gbeta) + ray.slot;
      AT(gb, 0) = f2.d[0];
      AT(gb, 1) = f2.d[1];
    }
  }
  AT(store, size_t(blockIdx.y) * per_img + in + lane) = double4{ray.x, ray.y, lx, ly};
}

// One deflector's (or, of TNFW, a pair's) sums over rays [r0, r1) of `st`: a
// lane per ray, each entry read once for the pair.
template <int D>
__device__ __forceinline__ void tnfw_sums(const double *const (&rd)[2], const double4 *st, int64_t r0, int64_t r1,
                                          int lane, double (&acc)[2][LENSIM_NPARAM]) {
  const TnfwRec ra(rd[0]), rb(rd[D - 1]);
  for (int64_t r = r0 + lane; r < r1; r += 64) {
    const double4 s = AT(st, r);
    if (s.z == 0.0 && s.w == 0.0) continue;
    tnfw_ray_grad(ra, rd[0], s.x, s.y, s.z, s.w, acc[0]);
    if constexpr (D == 2) tnfw_ray_grad(rb, rd[1], s.x, s.y, s.z, s.w, acc[1]);
  }
}

// Partial sums [img - img0][plane or bulk index][split][8] of lambda . d alpha /
// d kwargs over a round's rays, stored by the first round, to which the others
// add: a wave takes two planes' (or bulk) deflectors
// q, q + 1 and one of the splits of the rays.  SUBS: the subhalos and linear
// deflectors; REST: the others, whose duals' registers would cost those waves.
// A launch of one kind leaves the other's deflectors alone; a short list's two
// kinds go in one launch (4 us less a call).
template <typename T, bool HALO, bool SUBS, bool REST>
__global__ __launch_bounds__(256) void defl_grad_kernel(ModelArgs m, GridArgs g, GradArgs ga,
                                                        const double *__restrict__ recd,
                                                        const float *__restrict__ recf,
                                                        const double *__restrict__ coefd,
                                                        const float *__restrict__ coeff,
                                                        const int *__restrict__ tab_all,
                                                        const double4 *__restrict__ store, size_t per_img, int n,
                                                        int img0, int round, bool both,
                                                        double *__restrict__ gpart_mp) {
  const int img = img0 + blockIdx.y, lane = threadIdx.x & 63;
  if (!SUBS && both && m.mp_n && mp_tab(m, tab_all, img).sub) return;  // no such deflector
  const int q = 2 * __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (q >= n) return;
  const int nq = min(2, n - q);
  double *part = gpart_mp + ((size_t(blockIdx.y) * n + q) * gridDim.z + blockIdx.z) * LENSIM_NPARAM;  // of q; q + 1 after
  const size_t next = size_t(gridDim.z) * LENSIM_NPARAM;                                             // gridDim.z splits
  const RecPtrs<T> rp = rec_ptrs<T>(m, recd, recf, coefd, coeff, img);
  int k[2], type[2], run[2], runs = 1;
  if (m.mp_n) {
    const MpTab tab = mp_tab(m, tab_all, img);
    runs = tab.n;
    for (int d = 0; d < nq; ++d) {
      const int v = __builtin_amdgcn_readfirstlane(AT(tab.who, q + d));
      k[d] = v & ((1 << kWhoBits) - 1);
      type[d] = v >> kWhoBits;
      run[d] = __builtin_amdgcn_readfirstlane(AT(tab.run_of, q + d));
    }
  } else {
    for (int d = 0; d < nq; ++d) {
      k[d] = m.n_lens + q + d;
      type[d] = __builtin_amdgcn_readfirstlane(m.bulk_type ? m.bulk_type : AT(m.bulk_types, q + d));
      if (!bulk_type_ok_dev(type[d])) type[d] = LENSIM_NULL;
      run[d] = 0;
    }
  }
  // the round's rays and this split's share of them (whole waves)
  const int64_t cap = round_rays(per_img, runs), left = int64_t(g.nx) * g.ny * g.s * g.s - round * cap;
  const int64_t n_ray = left < 0 ? 0 : (left < cap ? left : cap);
  const int64_t len = ((n_ray + 63) / 64 + gridDim.z - 1) / gridDim.z * 64;
  const int64_t r0 = min(n_ray, len * blockIdx.z), r1 = min(n_ray, r0 + len);
  if (r0 == r1 && (SUBS || round)) {  // nothing of this round (REST's deflectors are stored over by its launch, after)
    if (!round && lane < nq * LENSIM_NPARAM) AT(part, lane / LENSIM_NPARAM * next + lane % LENSIM_NPARAM) = 0.0;
    return;
  }
  const double4 *st[2];
  const double *rd[2];
  for (int d = 0; d < 2; ++d) {
    st[d] = store + size_t(blockIdx.y) * per_img + size_t(run[d < nq ? d : 0]) * cap;
    rd[d] = rp.recd + k[d < nq ? d : 0] * kRec;
  }
  double acc[2][LENSIM_NPARAM];
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int i = 0; i < LENSIM_NPARAM; ++i) acc[d][i] = 0.0;
  const bool pair = nq == 2 && type[0] == LENSIM_TNFW && type[1] == LENSIM_TNFW && run[0] == run[1];
  if (SUBS && pair) {
    if constexpr (HALO) tnfw_sums<2>(rd, st[0], r0, r1, lane, acc);
  } else {
    for (int d = 0; d < nq; ++d) {
      double a[2][LENSIM_NPARAM];
#pragma unroll
      for (int i = 0; i < LENSIM_NPARAM; ++i) a[0][i] = 0.0;
      if (SUBS && type[d] == LENSIM_TNFW) {
        if constexpr (HALO) {
          const double *const r[2] = {rd[d], rd[d]};
          tnfw_sums<1>(r, st[d], r0, r1, lane, a);
        }
      } else if (SUBS && (type[d] == LENSIM_CONVERGENCE || type[d] == LENSIM_SHEAR)) {
        const double cx = rd[d][R_CX], cy = rd[d][R_CY], c2 = rd[d][2], c3 = rd[d][3];
        const bool conv = type[d] == LENSIM_CONVERGENCE;
        for (int64_t r = r0 + lane; r < r1; r += 64) {
          const double4 s = AT(st[d], r);
          if (s.z == 0.0 && s.w == 0.0) continue;
          const double dx = s.x - cx, dy = s.y - cy;
          if (conv) {  // alpha = kappa (dx, dy)
            a[0][0] += s.z * dx + s.w * dy;
            a[0][1] -= c2 * s.z;
            a[0][2] -= c2 * s.w;
          } else {  // alpha = (g1 dx + g2 dy, g2 dx - g1 dy)
            a[0][0] += s.z * dx - s.w * dy;
            a[0][1] += s.z * dy + s.w * dx;
            a[0][2] -= c2 * s.z + c3 * s.w;
            a[0][3] -= c3 * s.z - c2 * s.w;
          }
        }
      } else if (REST && !sub_type(type[d])) {
        for (int64_t r = r0 + lane; r < r1; r += 64) {
          const double4 s = AT(st[d], r);
          if (s.z == 0.0 && s.w == 0.0) continue;
          double ax = 0.0, ay = 0.0, dax[LENSIM_NPARAM], day[LENSIM_NPARAM], dcen[4];
          deflector_dalpha<T, HALO>(m, ga, rp, img, k[d], type[d], s.x, s.y, ax, ay, dax, day, dcen);
#pragma unroll
          for (int i = 0; i < LENSIM_NPARAM; ++i) a[0][i] += s.z * dax[i] + s.w * day[i];
        }
      }
#pragma unroll
      for (int i = 0; i < LENSIM_NPARAM; ++i) {
        if (d == 0) acc[0][i] = a[0][i];
        else acc[1][i] = a[0][i];
      }
    }
  }
  for (int d = 0; d < nq; ++d) {
    if (sub_type(type[d]) ? !SUBS : !REST) continue;
    double v[LENSIM_NPARAM];
#pragma unroll
    for (int i = 0; i < LENSIM_NPARAM; ++i) v[i] = wave_sum(d == 0 ? acc[0][i] : acc[1][i]);
    if (type[d] == LENSIM_TNFW) tnfw_grad_scale(rd[d], v);
    if (lane < LENSIM_NPARAM) {
      double mine = 0.0;
#pragma unroll
      for (int i = 0; i < LENSIM_NPARAM; ++i) mine = lane == i ? v[i] : mine;
      AT(part, d * next + lane) = round ? AT(part, d * next + lane) + mine : mine;
    }
  }
}

// A kwarg p of the list's deflector k of image img, summed over its splits
// (gpart_mp: image li of the part of the batch that it holds): lane j of eight
// takes the splits j, j + 8, ..., then the lanes' sums are added in pairs.  A
// deflector that the caller's order names on several planes gets the sum over
// them, one that it does not name zero; a model of more runs than the caller's
// bound, whose rays the plan's rounds did not all take, NaN.
__device__ __forceinline__ double list_sum(const ModelArgs &m, const int *tab_all, const double *gpart_mp, int n,
                                           int splits, int runs, int li, int img, int k, int p, int j) {
  double v = 0.0;
  auto add = [&](int q) {
    for (int b = j; b < splits; b += 8) v += AT(gpart_mp, ((size_t(li) * n + q) * splits + b) * LENSIM_NPARAM + p);
  };
  if (!m.mp_n) {
    add(k - m.n_lens);
  } else {
    const MpTab tab = mp_tab(m, tab_all, img);
    if (tab.n > runs) {
      v = NAN;
    } else if (!tab.dup) {
      if (AT(tab.plane_of, k) >= 0) add(AT(tab.plane_of, k));
    } else {
      for (int q = 0; q < n; ++q)
        if ((AT(tab.who, q) & ((1 << kWhoBits) - 1)) == k) add(q);
    }
  }
  for (int off = 8; off < 64; off <<= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// The list's sums of images img0 .. img0 + n_img - 1 (a part of the batch) into
// the first of the nblk slots grad_reduce_kernel reads, the others zero.
__global__ __launch_bounds__(256) void defl_partial_reduce(ModelArgs m, const int *__restrict__ tab_all,
                                                           const double *__restrict__ gpart_mp, int n, int splits,
                                                           int runs, int img0, int n_img, int nblk,
                                                           double *__restrict__ gpart) {
  const int k0 = m.mp_n ? 0 : m.n_lens, nk = m.n_defl - k0;
  const int64_t r = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (r >= int64_t(n_img) * nk) return;
  const int p = threadIdx.x & 7, j = (threadIdx.x >> 3) & 7, li = int(r / nk), k = k0 + int(r - int64_t(li) * nk);
  const double v = list_sum(m, tab_all, gpart_mp, n, splits, runs, li, img0 + li, k, p, j);
  const size_t o = (size_t(img0 + li) * m.n_prof + k) * nblk;
  for (int b = j; b < nblk; b += 8) AT(gpart, (o + b) * LENSIM_NPARAM + p) = b == 0 ? v : 0.0;
}

// The gradient of the multi-plane or bulk list into ga.gpart, and beta (and
// dS/dbeta) at every ray for the launches that follow.
template <typename T, bool HALO>
int launch_defl_grad(const ModelArgs &m, const GridArgs &g, const GradArgs &ga, const double *recd, const float *recf,
                     const int *tab, double *gpart_mp, double4 *store, int nblk, int n_img, hipStream_t st) {
  const size_t rays = size_t(g.nx) * g.ny * g.s * g.s;
  const DeflGradPlan p = defl_grad_plan(m, rays, n_img);
  // a round's rays (of several planes, as many as one run would leave): so a launch's threads stay below 2^32
  const size_t some = p.n && p.per_img < rays ? p.per_img : rays;
  int sub = sub_list(m);
  if (!m.mp_n && sub == 0) sub = m.bulk_type ? int(sub_type(m.bulk_type)) : 2;  // of the bulk list alone
  // of an inline list the types are known: a launch for the kinds it holds
  bool any_sub = m.n_bulk > 0;
  for (int k = 0; m.mp_n && k < m.n_lens; ++k) any_sub = any_sub || sub_type(m.types[k]);
  for (int i0 = 0; i0 < n_img; i0 += p.imgs) {
    const int ni = n_img - i0 < p.imgs ? n_img - i0 : p.imgs;
    const dim3 grid((unsigned)((some + 63) / 64), ni);
    const dim3 dgrid((p.n + 7) / 8, ni, p.splits);
    for (int r = 0; r < p.rounds; ++r) {
      if (!m.mp_n) {
        const bool kept = bulk_keeps<T>(m, size_t(g.nx) * g.ny);
        bulk_adjoint_kernel<T, HALO><<<grid, kept ? 64 : 64 * kBulkWaves, 0, st>>>(
            m, g, ga, recd, recf, ga.coefd, ga.coeff, store, p.per_img, i0, r, kept);
      } else {
        auto launch = [&](auto kernel, const MpLaunch &l) {
          kernel<<<l.grid, l.threads, 0, st>>>(m, g, ga, recd, recf, ga.coefd, ga.coeff, tab, sub == 2, store, p.per_img,
                                               i0, r, p.imgs >= n_img, m.mp_tij, m.mp_tz, m.mp_r2p);
        };
#define LENSIM_ADJOINT(H, S)                                                                          \
  do {                                                                                                \
    const MpLaunch l = mp_launch(m, rays, some, ni, S);                                               \
    launch(l.solo ? &mp_adjoint_kernel<T, H, S, true> : &mp_adjoint_kernel<T, H, S, false>, l);       \
  } while (0)
        if (sub) LENSIM_ADJOINT(true, true);
        if (sub != 1) LENSIM_ADJOINT(HALO, false);
#undef LENSIM_ADJOINT
      }
      int rc = check_launch("adjoint kernel");
      if (rc) return rc;
      if (p.n == 0) continue;  // no deflector: beta alone
      auto sums = [&](auto kernel) {
        kernel<<<dgrid, 256, 0, st>>>(m, g, ga, recd, recf, ga.coefd, ga.coeff, tab, store, p.per_img, p.n, i0, r,
                                      sub == 2, gpart_mp);
      };
      const bool rest = sub != 1;
      if (any_sub && rest && p.n <= 64) {
        sums(&defl_grad_kernel<T, HALO, true, true>);
      } else {
        if (any_sub) sums(&defl_grad_kernel<T, HALO, true, false>);
        if (rest) sums(&defl_grad_kernel<T, HALO, false, true>);
      }
      if ((rc = check_launch("defl_grad_kernel"))) return rc;
    }
    if (p.n == 0 || p.imgs >= n_img) continue;  // (grad_reduce_kernel adds up the batch's sums)
    const int64_t nw = int64_t(ni) * (m.n_defl - (m.mp_n ? 0 : m.n_lens));
    defl_partial_reduce<<<(unsigned)((nw + 3) / 4), 256, 0, st>>>(m, tab, gpart_mp, p.n, p.splits, p.runs, i0, ni, nblk,
                                                                  ga.gpart);
    const int rc = check_launch("defl_partial_reduce");
    if (rc) return rc;
  }
  return LENSIM_OK;
}

// The gradient from the profiles' partials, a thread each; the first
// list_blocks blocks: that of the list's deflectors from their splits, a wave
// each (0: they are in gpart, or there is no list).
__global__ __launch_bounds__(256) void grad_reduce_kernel(ModelArgs m, const int *__restrict__ tab_all,
                                                          const double *__restrict__ gpart_mp, DeflGradPlan pl,
                                                          int list_blocks, int n_img,
                                                          const double *__restrict__ gpart, int nblk,
                                                          double *__restrict__ grad) {
  const int k0 = m.mp_n ? 0 : m.n_lens, nk = m.n_defl - k0;
  if (int(blockIdx.x) < list_blocks) {
    const int64_t r = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (r >= int64_t(n_img) * nk) return;
    const int p = threadIdx.x & 7, j = (threadIdx.x >> 3) & 7, img = int(r / nk), k = k0 + int(r - int64_t(img) * nk);
    const double v = list_sum(m, tab_all, gpart_mp, pl.n, pl.splits, pl.runs, img, img, k, p, j);
    if (j == 0) AT(grad, (size_t(img) * m.n_prof + k) * LENSIM_NPARAM + p) = v;
    return;
  }
  const int idx = (blockIdx.x - list_blocks) * 256 + threadIdx.x;  // (img * n_prof + k) * 8 + q
  if (idx >= n_img * m.n_prof * LENSIM_NPARAM) return;
  const int q = idx % LENSIM_NPARAM, ik = idx / LENSIM_NPARAM, k = ik % m.n_prof;
  if (list_blocks && k >= k0 && k < m.n_defl) return;
  double s = 0.0;
  for (int b = 0; b < nblk; ++b) s += AT(gpart, (size_t(ik) * nblk + b) * LENSIM_NPARAM + q);
  AT(grad, idx) = s;
}

// One wave per image: lane l sums partials l, l + 64, ... and a fixed
// butterfly adds the 64 lane sums, so the order depends on n_tiles alone (not
// on the batch); the partials of an image are read contiguously.
// add: a term per image (the linear solve's marginalisation constant), or NULL.
__global__ __launch_bounds__(64) void logl_kernel(const double *__restrict__ partial, int n_tiles,
                                                  const double *__restrict__ add, double *__restrict__ logl) {
  const int img = blockIdx.x;
  const double *p = partial + size_t(img) * n_tiles;
  double s = 0.0;
  for (int t = threadIdx.x; t < n_tiles; t += 64) s += AT(p, t);
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (threadIdx.x == 0) AT(logl, img) = -s / 2.0 + (add ? AT(add, img) : 0.0);
}

// ------------------------------------------------------------ launches ---

int check_launch(const char *where) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, where);
  return LENSIM_OK;
}

int launch_prep(const ModelArgs &m, const double *params, int n_img, unsigned char *ws, const Layout &L,
                hipStream_t st, bool with_dcoef = false) {
  const int n = n_img * m.n_prof;
  if (n == 0) return LENSIM_OK;
  prep_kernel<<<(n + 63) / 64, 64, 0, st>>>(m, params, n_img, reinterpret_cast<double *>(ws + L.recd),
                                             reinterpret_cast<float *>(ws + L.recf),
                                             reinterpret_cast<double *>(ws + L.coefd),
                                             reinterpret_cast<float *>(ws + L.coeff),
                                             with_dcoef ? reinterpret_cast<double *>(ws + L.dcoefd) : nullptr,
                                             with_dcoef ? reinterpret_cast<float *>(ws + L.dcoeff) : nullptr);
  return check_launch("prep_kernel");
}

int grid_args(const lensim_grid *grid, GridArgs &g) {
  if (!grid) return fail(LENSIM_EINVAL, "grid is NULL");
  if (grid->nx <= 0 || grid->ny <= 0 || grid->supersampling <= 0)
    return fail(LENSIM_EINVAL, "grid sizes must be positive (nx=%d ny=%d s=%d)", grid->nx, grid->ny,
                grid->supersampling);
  if (int64_t(grid->nx) * grid->ny > (int64_t(1) << 30)) return fail(LENSIM_EINVAL, "grid too large");
  g.nx = grid->nx;
  g.ny = grid->ny;
  g.s = grid->supersampling;
  g.ra0 = grid->ra_at_xy_0;
  g.dec0 = grid->dec_at_xy_0;
  g.m00 = grid->pix2angle[0];
  g.m01 = grid->pix2angle[1];
  g.m10 = grid->pix2angle[2];
  g.m11 = grid->pix2angle[3];
  const double det = g.m00 * g.m11 - g.m01 * g.m10;
  const double pixel_width = sqrt(fabs(det));  // lenstronomy PixelGrid.pixel_width
  g.scale = pixel_width * pixel_width / (double(g.s) * double(g.s));
  g.mask = grid->d_eval_mask;
  g.mask_nx = g.nx;
  g.mask_s = 1;
  grid_consts(g);
  return LENSIM_OK;
}

// The model with the sub-ray steps of grid g (SubSteps) for its records.
ModelArgs with_grid(const ModelArgs &m, const GridArgs &g) {
  ModelArgs mg = m;
  const double inv_s = 1.0 / g.s;
  mg.sub.sx[0] = g.m00 * inv_s;
  mg.sub.sx[1] = g.m10 * inv_s;
  mg.sub.rr[0] = g.m01 * inv_s - g.s * mg.sub.sx[0];
  mg.sub.rr[1] = g.m11 * inv_s - g.s * mg.sub.sx[1];
  mg.sub.asc = m.alpha_scaling;
  return mg;
}

int psf_dims(const lensim_psf *psf, uint32_t flags, int &kx, int &ky, int &edge) {
  const bool none = !psf || psf->type == LENSIM_PSF_NONE || (flags & LENSIM_IMAGE_UNCONVOLVED);
  if (none) {
    kx = ky = 1;
    edge = 0;
    return LENSIM_OK;
  }
  if (psf->type != LENSIM_PSF_PIXEL && psf->type != LENSIM_PSF_GAUSSIAN)
    return fail(LENSIM_EUNSUPPORTED, "psf type %d not supported", psf->type);
  if (psf->kx <= 0 || psf->ky <= 0 || !(psf->kx & 1) || !(psf->ky & 1))
    return fail(LENSIM_EINVAL, "psf kernel must have odd positive sizes (got %d x %d)", psf->ky, psf->kx);
  if (!psf->d_kernel) return fail(LENSIM_EINVAL, "psf kernel pointer is NULL");
  kx = psf->kx;
  ky = psf->ky;
  edge = psf->type == LENSIM_PSF_GAUSSIAN;
  return LENSIM_OK;
}

// Supersampled-convolution plan of a PSF on grid g (off when unconvolved,
// without a PSF, or when the grid is not supersampled).
int psf_ss(const lensim_psf *psf, const GridArgs &g, uint32_t flags, SSPlan &ss) {
  ss = SSPlan();
  const bool none = !psf || psf->type == LENSIM_PSF_NONE || (flags & LENSIM_IMAGE_UNCONVOLVED);
  if (none || !psf->supersampled || g.s == 1) return LENSIM_OK;
  if (psf->supersampled != 1) return fail(LENSIM_EINVAL, "psf.supersampled must be 0 or 1");
  if (int64_t(g.nx) * g.ny * g.s * g.s > (int64_t(1) << 30)) return fail(LENSIM_EINVAL, "supersampled grid too large");
  ss.on = 1;
  ss.s = g.s;
  if (psf->kx_low || psf->ky_low || psf->d_kernel_low) {
    if (psf->type != LENSIM_PSF_PIXEL) return fail(LENSIM_EINVAL, "a split kernel needs a PIXEL psf");
    if (psf->kx_low <= 0 || psf->ky_low <= 0 || !(psf->kx_low & 1) || !(psf->ky_low & 1))
      return fail(LENSIM_EINVAL, "low-resolution kernel must have odd positive sizes (got %d x %d)", psf->ky_low,
                  psf->kx_low);
    if (!psf->d_kernel_low) return fail(LENSIM_EINVAL, "low-resolution kernel pointer is NULL");
    ss.kxl = psf->kx_low;
    ss.kyl = psf->ky_low;
  }
  return LENSIM_OK;
}

template <typename T>
size_t conv_smem(int kx, int kyp, int ty = ConvTile<T>::TY) {
  return size_t((ty + kyp - 1) | 1) * (ConvTile<T>::TX + kx - 1) * sizeof(T);
}

// conv_kernel over n_img images (c.n_tiles_x is set here, the tile count goes
// to *n_tiles): 64-row tiles where their LDS fits (four waves a block, a
// smaller share of halo rows), 32-row tiles otherwise.  FP64 images go to
// conv_f64_kernel as long as its tile fits the LDS.
template <typename T, int TY, bool LW, int CLS = 0>
int launch_conv_tile(const ConvArgs &c, dim3 grid, size_t smem, const T *in, const double *kf, T *out,
                     double *partial, hipStream_t st) {
  if (smem > 65536) {  // dynamic LDS beyond 64 KB needs the kernel attribute raised first
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&conv_kernel<T, TY, LW, CLS>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, int(smem));
    if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(conv_kernel)");
  }
  conv_kernel<T, TY, LW, CLS><<<grid, ConvTile<T>::TX * TY / kWin, smem, st>>>(c, in, kf, out, partial);
  return check_launch("conv_kernel");
}

template <int R, int H, int CLS, bool GW>
int launch_conv_f64(ConvArgs c, int n_img, const double *in, const double *kf, double *out, double *partial,
                    int *n_tiles, hipStream_t st) {
  const size_t smem = conv_f64_smem(c.kx, c.ky, R, H, CLS, GW);
  c.n_tiles_x = (c.nx + 31) / 32;
  *n_tiles = c.n_tiles_x * ((c.ny + 15) / 16);
  if (smem > 65536) {  // dynamic LDS beyond 64 KB needs the kernel attribute raised first
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&conv_f64_kernel<R, H, CLS, GW>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, int(smem));
    if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(conv_f64_kernel)");
  }
  const dim3 grid(c.n_tiles_x * ((c.ny + 2 * R * H - 1) / (2 * R * H)), n_img);
  conv_f64_kernel<R, H, CLS, GW><<<grid, 64 * CLS * H, smem, st>>>(c, conv_f64_rows(c.ky, R, H), in, kf, out, partial);
  return check_launch("conv_f64_kernel");
}

template <typename T>
int launch_conv_kernel(ConvArgs c, int n_img, const T *in, const double *kf, T *out, double *partial,
                       int *n_tiles, hipStream_t st) {
  if constexpr (sizeof(T) == sizeof(double)) {
    // Classes of kernel columns by the kernel alone, so that an image's sums are
    // the same in any batch: below ten columns the split's barriers cost more
    // than the work it shares (5 x 5, 64 images of 180^2, 57.5 against 67.7 us a
    // call; one image of 60^2 with 11 x 11 19.4 with, 21.5 without).  The shape
    // by the number of 32 x 32 tiles and the LDS: with fewer tiles than CUs short
    // ones, weights in LDS; from eight a CU (2048 tiles) kernels below 16 x 16 go
    // to conv_kernel in the same order, whose waves hold fewer registers (64
    // images of 180^2 with 15 x 15 74.6 against 80.4 us a call, 128 120.8 against
    // 145; at 1024 tiles, 256 of 60^2, 46.5 against 43.9).  One block of 82 KB
    // LDS or more fills a CU: there two row groups of waves (81 x 81, 743 against
    // 918 us).
    const size_t tiles = size_t((c.nx + 31) / 32) * ((c.ny + 31) / 32) * n_img;
    const bool few = tiles < size_t(cu_count());
    auto fits = [&](int r, int h, int cls, bool gw, size_t lds) {
      return conv_f64_smem(c.kx, c.ky, r, h, cls, gw) <= lds;
    };
    if (c.kx < 16 && c.ky < 16 && tiles >= 8 * size_t(cu_count())) {
      c.n_tiles_x = (c.nx + 31) / 32;
      *n_tiles = c.n_tiles_x * ((c.ny + 15) / 16);
      const dim3 grid(c.n_tiles_x * ((c.ny + 63) / 64), n_img);
      const size_t smem = conv_smem<T>(c.kx, c.kyp, 64);
      return c.kx < 10 ? launch_conv_tile<T, 64, false, 1>(c, grid, smem, in, kf, out, partial, st)
                       : launch_conv_tile<T, 64, false, 4>(c, grid, smem, in, kf, out, partial, st);
    }
#define LENSIM_CONV(R, H, CLS, GW) launch_conv_f64<R, H, CLS, GW>(c, n_img, in, kf, out, partial, n_tiles, st)
    if (c.kx < 10 && fits(8, 4, 1, true, kMaxLds / 2) && fits(4, 4, 1, false, kMaxLds))
      return LENSIM_CONV(4, 4, 1, false);
    // (a wide flat kernel whose tall tiles do not fit stays with conv_kernel in any batch)
    const bool one = fits(16, 1, 4, true, kMaxLds / 2), two = fits(16, 2, 4, true, kMaxLds);
    if (few && (one || two) && fits(4, 2, 4, false, kMaxLds)) return LENSIM_CONV(4, 2, 4, false);
    if (one) return LENSIM_CONV(16, 1, 4, true);
    if (two) return LENSIM_CONV(16, 2, 4, true);
#undef LENSIM_CONV
  }
  constexpr int TX = ConvTile<T>::TX;
  int ty = ConvTile<T>::TY;
  if (conv_smem<T>(c.kx, c.kyp, 64) <= kMaxLds) ty = 64;
  c.n_tiles_x = (c.nx + TX - 1) / TX;
  *n_tiles = c.n_tiles_x * ((c.ny + ty - 1) / ty);
  const size_t smem = conv_smem<T>(c.kx, c.kyp, ty);
  if (smem > kMaxLds) return fail(LENSIM_EUNSUPPORTED, "psf %dx%d needs %zu B of LDS per tile", c.ky, c.kx, smem);
  const dim3 grid(*n_tiles, n_img);
  // weights in LDS when the launch has fewer blocks than the GPU has CUs
  const size_t smem_lw = ((smem + 7) & ~size_t(7)) + size_t(c.kx) * c.kyp * sizeof(double);
  const bool lw = size_t(*n_tiles) * n_img < 256 && smem_lw <= kMaxLds;
  if (ty == 64)
    return lw ? launch_conv_tile<T, 64, true>(c, grid, smem_lw, in, kf, out, partial, st)
              : launch_conv_tile<T, 64, false>(c, grid, smem, in, kf, out, partial, st);
  return lw ? launch_conv_tile<T, ConvTile<T>::TY, true>(c, grid, smem_lw, in, kf, out, partial, st)
            : launch_conv_tile<T, ConvTile<T>::TY, false>(c, grid, smem, in, kf, out, partial, st);
}

// Whether the mixed form convolves on the matrix cores (any real PSF whose
// MFMA tile fits in 64 KB of LDS) or on the vector ALUs.
template <typename T>
bool use_mfma(bool identity, int kx, int ky) {
  if (sizeof(T) != sizeof(float) || identity) return false;
  return mfma_nks(kx) <= kMfMaxNks && mfma_smem(kx, ky, 2) <= kMaxLds;
}

template <int NKS, int TL>
int launch_conv_mfma_n(const ConvArgs &c, dim3 grid, const float *in, const int *hdr, const half8 *frag,
                       const float *blkmax, int nblk, float *out, double *partial, hipStream_t st) {
  const size_t smem = mfma_smem(c.kx, c.ky, TL);
  if (smem > 65536) {  // dynamic LDS beyond 64 KB needs the kernel attribute raised first
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&conv_mfma_kernel<NKS, TL>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, int(smem));
    if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(conv_mfma_kernel)");
  }
  conv_mfma_kernel<NKS, TL><<<grid, 256, smem, st>>>(c, mfma_ls(c.kx, TL), in, hdr, frag, blkmax, nblk, out,
                                                      partial);
  return check_launch("conv_mfma_kernel");
}

template <int NKS>
int launch_conv_mfma_tl(const ConvArgs &c, int tl, dim3 grid, const float *in, const int *hdr, const half8 *frag,
                        const float *blkmax, int nblk, float *out, double *partial, hipStream_t st) {
  switch (tl) {
    case 2: return launch_conv_mfma_n<NKS, 2>(c, grid, in, hdr, frag, blkmax, nblk, out, partial, st);
    case 3: return launch_conv_mfma_n<NKS, 3>(c, grid, in, hdr, frag, blkmax, nblk, out, partial, st);
    case 4: return launch_conv_mfma_n<NKS, 4>(c, grid, in, hdr, frag, blkmax, nblk, out, partial, st);
    default: return fail(LENSIM_EINVAL, "matrix-core tile width %d", tl);
  }
}

// The MFMA convolution of n_img images by plan pl (c.kx, c.ky, c.edge set;
// c.n_tiles_x is set here).
int launch_conv_mfma(ConvArgs c, const MfmaPlan &pl, int n_img, const float *in, const int *hdr, const half8 *frag,
                     const float *blkmax, int nblk, float *out, double *partial, hipStream_t st) {
  if (pl.tl == 0) return fail(LENSIM_EUNSUPPORTED, "psf %dx%d exceeds the matrix-core tile's LDS", c.ky, c.kx);
  c.n_tiles_x = pl.n_tiles_x;
  const dim3 grid(pl.n_tiles, n_img);
  switch (mfma_nks(c.kx)) {
    case 1: return launch_conv_mfma_tl<1>(c, pl.tl, grid, in, hdr, frag, blkmax, nblk, out, partial, st);
    case 2: return launch_conv_mfma_tl<2>(c, pl.tl, grid, in, hdr, frag, blkmax, nblk, out, partial, st);
    case 3: return launch_conv_mfma_tl<3>(c, pl.tl, grid, in, hdr, frag, blkmax, nblk, out, partial, st);
    case 4: return launch_conv_mfma_tl<4>(c, pl.tl, grid, in, hdr, frag, blkmax, nblk, out, partial, st);
    default: return fail(LENSIM_EUNSUPPORTED, "psf width %d exceeds the matrix-core convolution", c.kx);
  }
}

// The PSF preparation of a call on the grid itself, and which convolution it is
// for.
template <typename T>
struct ConvChoice {
  bool mfma;
  PsfJob job;
  ConvChoice(const lensim_psf *psf, unsigned flags, int kx, int ky, unsigned char *ws, const Layout &L) {
    const bool identity = !psf || psf->type == LENSIM_PSF_NONE || (flags & LENSIM_IMAGE_UNCONVOLVED);
    mfma = use_mfma<T>(identity, kx, ky);
    job = PsfJob{};
    job.mode = mfma ? 2 : 1;
    job.k = identity ? nullptr : psf->d_kernel;
    job.kx = kx;
    job.ky = ky;
    job.kyp = kyp_of(ky);
    job.kt = reinterpret_cast<double *>(ws + L.psf);
    job.hdr = reinterpret_cast<int *>(ws + L.bfrag);
    job.frag = reinterpret_cast<half8 *>(ws + L.bfrag + 16);
    if (mfma) {
      job.nks = mfma_nks(kx);
      job.n_steps = mfma_steps(kx, ky);
    }
  }
};

// The records (with EPL coefficients' derivatives when dc), the PSF
// preparation and the runs of up to kMpPrep planes in one launch (4 us less a call
// of a few deflectors); the runs of more, which want a block's 1024 threads, in
// another.
int launch_prep_psf(const ModelArgs &m, const double *params, int n_img, const PsfJob &pj, bool dc, unsigned char *ws,
                    const Layout &L, hipStream_t st) {
  const int nb_prep = (n_img * m.n_prof + 255) / 256;
  const int nb_runs = m.mp_n > 0 && m.mp_n <= kMpPrep ? int(mp_tab_sets(m, n_img)) : 0;
  int *tab = reinterpret_cast<int *>(ws + L.mp_tab);
  prep_psf_kernel<<<nb_prep + nb_runs + psf_job_blocks(pj), 256, 0, st>>>(
      m, params, n_img, reinterpret_cast<double *>(ws + L.recd), reinterpret_cast<float *>(ws + L.recf),
      reinterpret_cast<double *>(ws + L.coefd), reinterpret_cast<float *>(ws + L.coeff),
      dc ? reinterpret_cast<double *>(ws + L.dcoefd) : nullptr, dc ? reinterpret_cast<float *>(ws + L.dcoeff) : nullptr,
      pj, tab, nb_prep, nb_runs);
  int rc = check_launch("prep_psf_kernel");
  if (!rc && m.mp_n > 0 && !nb_runs) rc = launch_mp_runs(m, tab, n_img, st);
  return rc;
}

// 'Same' convolution of n_img pooled images with the prepared PSF; with data
// in c also their chi^2 partials (n_tiles an image).
template <typename T>
int launch_conv(const ConvArgs &c, const ConvChoice<T> &cc, int n_img, const T *in, const float *blkmax, T *out,
                double *partial, int *n_tiles, hipStream_t st) {
  if (!cc.mfma) return launch_conv_kernel<T>(c, n_img, in, cc.job.kt, out, partial, n_tiles, st);
  *n_tiles = n16_tiles(c.nx, c.ny);  // chi^2 partials of the 16 x 16 output tiles
  return launch_conv_mfma(c, mfma_plan(c.nx, c.ny, n_img, c.kx, c.ky), n_img, reinterpret_cast<const float *>(in),
                          cc.job.hdr, cc.job.frag, blkmax, (c.nx * c.ny + 255) / 256, reinterpret_cast<float *>(out),
                          partial, st);
}

// The image pipeline shared by lensim_image and lensim_loglike.
template <typename T>
int run_image(const ModelArgs &m_in, const GridArgs &g, const lensim_psf *psf, int kx, int ky, int edge,
              const lensim_data *data, const double *params, int n_img, unsigned flags, T *out, double *logl,
              unsigned char *ws, const Layout &L, hipStream_t st, T *gout = nullptr,
              const MpKeep &keep = MpKeep{}) {
  const ModelArgs m = with_grid(m_in, g);
  const ConvChoice<T> cc(psf, flags, kx, ky, ws, L);
  int rc = launch_prep_psf(m, params, n_img, cc.job, gout != nullptr, ws, L, st);
  if (rc) return rc;
  T *lowres = reinterpret_cast<T *>(ws + L.lowres);
  float *blkmax = cc.mfma ? reinterpret_cast<float *>(ws + L.blkmax) : nullptr;
  const int *tab = reinterpret_cast<const int *>(ws + L.mp_tab);
  timing_mark(0, st);
  const double *recd = reinterpret_cast<const double *>(ws + L.recd);
  const float *recf = reinterpret_cast<const float *>(ws + L.recf);
  const double *coefd = reinterpret_cast<const double *>(ws + L.coefd);
  const float *coeff = reinterpret_cast<const float *>(ws + L.coeff);
  rc = launch_render<T>(m, g, recd, recf, coefd, coeff, tab, flags, keep, lowres, blkmax, n_img, st);
  if (rc) return rc;
  timing_mark(1, st);
  ConvArgs c{};
  c.nx = g.nx;
  c.ny = g.ny;
  c.kx = kx;
  c.ky = ky;
  c.kyp = cc.job.kyp;
  c.edge = edge;
  double *partial = nullptr;
  if (data) {
    c.data = data->d_data;
    c.noise = data->d_noise_map;
    c.expo = data->d_exposure_map;
    c.mask = data->d_mask;
    c.exposure_time = data->exposure_time;
    c.bkg2 = data->background_rms * data->background_rms;
    c.inv_t = 1.0 / data->exposure_time;
    c.gout = gout;
    c.dstride = data->image_stride;
    partial = reinterpret_cast<double *>(ws + L.partial);
  }
  int n_tiles;
  rc = launch_conv<T>(c, cc, n_img, lowres, blkmax, out, partial, &n_tiles, st);
  if (rc) return rc;
  timing_mark(2, st);
  if (data) {
    logl_kernel<<<n_img, 64, 0, st>>>(partial, n_tiles, nullptr, logl);
    rc = check_launch("logl_kernel");
    if (rc) return rc;
  }
  return LENSIM_OK;
}

// s x s block means of [n_img][ny s][nx s] into [n_img][ny][nx]
// (Util/image_util.py re_size).
template <typename T>
__global__ void pool_kernel(const T *__restrict__ in, int nx, int ny, int s, T *__restrict__ out) {
  const int pix = blockIdx.x * blockDim.x + threadIdx.x;
  if (pix >= nx * ny) return;
  const int img = blockIdx.y;
  const int y = pix / nx, x = pix - y * nx;
  const int nxh = nx * s;
  const T *src = in + size_t(img) * nx * ny * s * s + size_t(y) * s * nxh + size_t(x) * s;
  double acc = 0.0;
  for (int sy = 0; sy < s; ++sy)
    for (int sx = 0; sx < s; ++sx) acc += double(AT(src, size_t(sy) * nxh + sx));
  AT(out, size_t(img) * nx * ny + pix) = T(acc / (double(s) * double(s)));
}

// Final image of a supersampled convolution: the s x s mean of the convolved
// ray fluxes plus the low-resolution part (if any), with the chi^2 of every
// pixel reduced to one partial per block.
template <typename T>
__global__ __launch_bounds__(256) void combine_kernel(ConvArgs c, const T *__restrict__ chr, const T *__restrict__ lowc,
                                                      int s, T *__restrict__ out, double *__restrict__ partial) {
  const int img = blockIdx.y;
  const int npix = c.nx * c.ny;
  const int pix = blockIdx.x * blockDim.x + threadIdx.x;
  double chi = 0.0;
  if (pix < npix) {
    const int y = pix / c.nx, x = pix - y * c.nx;
    const int nxh = c.nx * s;
    const T *src = chr + size_t(img) * npix * s * s + size_t(y) * s * nxh + size_t(x) * s;
    double acc = 0.0;
    for (int sy = 0; sy < s; ++sy)
      for (int sx = 0; sx < s; ++sx) acc += double(AT(src, size_t(sy) * nxh + sx));
    double v = acc / (double(s) * double(s));
    if (lowc) v += double(AT(lowc, size_t(img) * npix + pix));
    const T m = T(v);
    if (out) AT(out, size_t(img) * npix + pix) = m;
    if (partial) chi = chi2_pixel<T>(c, pix, m, img);
    if (c.gout) AT(static_cast<T *>(c.gout), size_t(img) * npix + pix) = T(dlogl_dm(c, pix, double(m), img));
  }
  if (partial) {
    __shared__ double red[4];
    for (int off = 32; off > 0; off >>= 1) chi += __shfl_xor(chi, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = chi;
    __syncthreads();
    if (threadIdx.x == 0) AT(partial, size_t(img) * gridDim.x + blockIdx.x) = red[0] + red[1] + red[2] + red[3];
  }
}

// chi^2 of given model images, one partial per block of 256 pixels.
template <typename T>
__global__ __launch_bounds__(256) void data_chi2_kernel(ConvArgs c, const T *__restrict__ model,
                                                        double *__restrict__ partial) {
  const int img = blockIdx.y;
  const int npix = c.nx * c.ny;
  const int pix = blockIdx.x * blockDim.x + threadIdx.x;
  double chi = 0.0;
  if (pix < npix) chi = chi2_pixel<T>(c, pix, AT(model, size_t(img) * npix + pix), img);
  __shared__ double red[4];
  for (int off = 32; off > 0; off >>= 1) chi += __shfl_xor(chi, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = chi;
  __syncthreads();
  if (threadIdx.x == 0) AT(partial, size_t(img) * gridDim.x + blockIdx.x) = red[0] + red[1] + red[2] + red[3];
}

// Launches conv_kernel<T> ('same', zero or edge padding) of [n_img][ny][nx]
// with a prepared transposed kernel, no chi^2.
template <typename T>
int launch_conv_plain(int nx, int ny, int kx, int ky, int edge, const T *in, const double *kf, T *out, int n_img,
                      hipStream_t st) {
  ConvArgs c{};
  c.nx = nx;
  c.ny = ny;
  c.kx = kx;
  c.ky = ky;
  c.kyp = kyp_of(ky);
  c.edge = edge;
  int n_tiles = 0;
  return launch_conv_kernel<T>(c, n_img, in, kf, out, nullptr, &n_tiles, st);
}

// The rays of grid g as a grid of their own: pixel (I, J) is sub-ray
// (I mod s, J mod s) of pixel (I / s, J / s) (make_subgrid offsets), with the
// pixel_width^2 scale because the s x s mean follows the convolution.
GridArgs ray_grid(const GridArgs &g) {
  const int s = g.s;
  GridArgs gh = g;
  const double o0 = -0.5 + 1.0 / (2.0 * s);
  gh.nx = g.nx * s;
  gh.ny = g.ny * s;
  gh.s = 1;
  gh.ra0 = g.ra0 + (g.m00 + g.m01) * o0;
  gh.dec0 = g.dec0 + (g.m10 + g.m11) * o0;
  gh.m00 = g.m00 / s;
  gh.m01 = g.m01 / s;
  gh.m10 = g.m10 / s;
  gh.m11 = g.m11 / s;
  gh.scale = g.scale * double(s) * double(s);
  gh.mask_s = g.mask_s * s;
  grid_consts(gh);
  return gh;
}

// Adjoint of the s x s mean: out[J][I] (+)= in[J / s][I / s] / s^2.
template <typename T>
__global__ void unpool_kernel(const T *__restrict__ in, int nx, int ny, int s, int accumulate, T *__restrict__ out) {
  const int nxh = nx * s, nyh = ny * s;
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= nxh * nyh) return;
  const int img = blockIdx.y;
  const int J = idx / nxh, I = idx - J * nxh;
  const double v = double(AT(in, size_t(img) * nx * ny + size_t(J / s) * nx + I / s)) / (double(s) * double(s));
  T &o = AT(out, size_t(img) * nxh * nyh + idx);
  o = accumulate ? T(double(o) + v) : T(v);
}

// Supersampled convolution (supersampling_convolution=True,
// ImSim/Numerics/numerics.py:103-116, convolution.py:154-166, :238-252): the
// rays are rendered as a (ny s) x (nx s) image (each ray its own pixel),
// convolved there with the supersampled kernel, averaged over s x s, and the
// low-resolution split kernel's convolution of the averaged unconvolved rays
// is added.
template <typename T>
int run_image_ss(const ModelArgs &m_in, const GridArgs &g, const lensim_psf *psf, int kx, int ky, int edge,
                 const SSPlan &ss, const lensim_data *data, const double *params, int n_img, unsigned flags, T *out,
                 double *logl, unsigned char *ws, const Layout &L, hipStream_t st, T *gout = nullptr,
                 const MpKeep &keep = MpKeep{}) {
  const int s = ss.s;
  const GridArgs gh = ray_grid(g);
  const ModelArgs m = with_grid(m_in, gh);
  int rc = launch_prep(m, params, n_img, ws, L, st, gout != nullptr);
  if (rc) return rc;
  const bool mfma = use_mfma<T>(false, kx, ky);
  const int kyp = kyp_of(ky);
  double *kf = reinterpret_cast<double *>(ws + L.psf);
  int *hdr = reinterpret_cast<int *>(ws + L.bfrag);
  half8 *frag = reinterpret_cast<half8 *>(ws + L.bfrag + 16);
  if (mfma) {
    const int n_frag = mfma_steps(kx, ky) * 2 * 64;
    psf_mfma_prep_kernel<<<(n_frag + 255) / 256, 256, 0, st>>>(psf->d_kernel, kx, ky, mfma_nks(kx),
                                                               mfma_steps(kx, ky), hdr, frag);
    rc = check_launch("psf_mfma_prep_kernel");
  } else {
    psf_prep_kernel<<<(kyp * kx + 255) / 256, 256, 0, st>>>(psf->d_kernel, kx, ky, kyp, kf);
    rc = check_launch("psf_prep_kernel");
  }
  if (rc) return rc;
  const int npix = g.nx * g.ny, npix_h = gh.nx * gh.ny;
  T *hr = reinterpret_cast<T *>(ws + L.hr);
  T *chr = reinterpret_cast<T *>(ws + L.chr);
  float *blkmax = mfma ? reinterpret_cast<float *>(ws + L.blkmax) : nullptr;
  const double *recd = reinterpret_cast<const double *>(ws + L.recd);
  const float *recf = reinterpret_cast<const float *>(ws + L.recf);
  const double *coefd = reinterpret_cast<const double *>(ws + L.coefd);
  const float *coeff = reinterpret_cast<const float *>(ws + L.coeff);
  int *tab = reinterpret_cast<int *>(ws + L.mp_tab);
  if (m.mp_n && (rc = launch_mp_runs(m, tab, n_img, st))) return rc;
  timing_mark(0, st);
  rc = launch_render<T>(m, gh, recd, recf, coefd, coeff, tab, flags, keep, hr, blkmax, n_img, st);
  if (rc) return rc;
  timing_mark(1, st);
  if (mfma) {
    ConvArgs c{};
    c.nx = gh.nx;
    c.ny = gh.ny;
    c.kx = kx;
    c.ky = ky;
    c.kyp = kyp;
    c.edge = edge;
    rc = launch_conv_mfma(c, mfma_plan(gh.nx, gh.ny, n_img, kx, ky), n_img, reinterpret_cast<const float *>(hr),
                          hdr, frag, blkmax, (npix_h + 255) / 256, reinterpret_cast<float *>(chr), nullptr, st);
  } else {
    rc = launch_conv_plain<T>(gh.nx, gh.ny, kx, ky, edge, hr, kf, chr, n_img, st);
  }
  if (rc) return rc;
  T *lowc = nullptr;
  if (ss.kxl > 0) {
    T *lowu = reinterpret_cast<T *>(ws + L.lowu);
    lowc = reinterpret_cast<T *>(ws + L.lowc);
    double *kfl = reinterpret_cast<double *>(ws + L.psf_low);
    pool_kernel<T><<<dim3((npix + 255) / 256, n_img), 256, 0, st>>>(hr, g.nx, g.ny, s, lowu);
    if ((rc = check_launch("pool_kernel"))) return rc;
    const int kypl = kyp_of(ss.kyl);
    psf_prep_kernel<<<(kypl * ss.kxl + 255) / 256, 256, 0, st>>>(psf->d_kernel_low, ss.kxl, ss.kyl, kypl, kfl);
    if ((rc = check_launch("psf_prep_kernel (low)"))) return rc;
    if ((rc = launch_conv_plain<T>(g.nx, g.ny, ss.kxl, ss.kyl, 0, lowu, kfl, lowc, n_img, st))) return rc;
  }
  timing_mark(2, st);
  ConvArgs cc{};
  cc.nx = g.nx;
  cc.ny = g.ny;
  double *partial = nullptr;
  if (data) {
    cc.data = data->d_data;
    cc.noise = data->d_noise_map;
    cc.expo = data->d_exposure_map;
    cc.mask = data->d_mask;
    cc.exposure_time = data->exposure_time;
    cc.bkg2 = data->background_rms * data->background_rms;
    cc.inv_t = 1.0 / data->exposure_time;
    cc.dstride = data->image_stride;
    cc.gout = gout;
    partial = reinterpret_cast<double *>(ws + L.partial);
  }
  const int nblk = (npix + 255) / 256;
  combine_kernel<T><<<dim3(nblk, n_img), 256, 0, st>>>(cc, chr, lowc, s, out, partial);
  if ((rc = check_launch("combine_kernel"))) return rc;
  if (data) {
    logl_kernel<<<n_img, 64, 0, st>>>(partial, nblk, nullptr, logl);
    return check_launch("logl_kernel");
  }
  return LENSIM_OK;
}

// Zero-padded copy of [n_img][ny][nx] into [n_img][ny + 2 cy][nx + 2 cx].
template <typename T>
__global__ void pad_kernel(const T *__restrict__ in, int nx, int ny, int cx, int cy, T *__restrict__ out) {
  const int nxe = nx + 2 * cx, nye = ny + 2 * cy;
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= nxe * nye) return;
  const int img = blockIdx.y;
  const int Y = idx / nxe, X = idx - Y * nxe;
  const int y = Y - cy, x = X - cx;
  const T v = (y >= 0 && y < ny && x >= 0 && x < nx) ? AT(in, size_t(img) * nx * ny + size_t(y) * nx + x) : T(0);
  AT(out, size_t(img) * nxe * nye + idx) = v;
}

// Adjoint of edge clamping: pixel (y, x) receives every extended pixel
// (Y, X) with clamp(Y - cy) = y and clamp(X - cx) = x.
template <typename T>
__global__ void fold_kernel(const T *__restrict__ ext, int nx, int ny, int cx, int cy, T *__restrict__ out) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= nx * ny) return;
  const int img = blockIdx.y;
  const int y = idx / nx, x = idx - y * nx;
  const int nxe = nx + 2 * cx, nye = ny + 2 * cy;
  const int y0 = y == 0 ? 0 : y + cy, y1 = y == ny - 1 ? nye - 1 : y + cy;
  const int x0 = x == 0 ? 0 : x + cx, x1 = x == nx - 1 ? nxe - 1 : x + cx;
  const T *e = ext + size_t(img) * nxe * nye;
  double s = 0.0;
  for (int Y = y0; Y <= y1; ++Y)
    for (int X = x0; X <= x1; ++X) s += double(AT(e, size_t(Y) * nxe + X));
  AT(out, size_t(img) * nx * ny + idx) = T(s);
}

// Adjoint of the 'same' convolution of [n_img][ny][nx] by a kernel prepared
// UNflipped in kf (a correlation): zero padding directly; edge padding via the
// extended domain.  The forward pass with edge padding is a valid correlation
// of the edge-extended image E[Y][X] = in[clamp(Y - cy)][clamp(X - cx)], so its
// adjoint is the zero-padded 'same' correlation over the extended domain,
// folded back onto the pixels each extended one copies.
template <typename T>
int adjoint_conv(int nx, int ny, int kx, int ky, int edge, const T *gin, const double *kf, T *gout, T *gpad, T *gext,
                 int n_img, hipStream_t st) {
  if (!edge) return launch_conv_plain<T>(nx, ny, kx, ky, 0, gin, kf, gout, n_img, st);
  const int cx = (kx - 1) / 2, cy = (ky - 1) / 2;
  const int nxe = nx + 2 * cx, nye = ny + 2 * cy;
  const int ne = nxe * nye;
  pad_kernel<T><<<dim3((ne + 255) / 256, n_img), 256, 0, st>>>(gin, nx, ny, cx, cy, gpad);
  int rc = check_launch("pad_kernel");
  if (rc) return rc;
  if ((rc = launch_conv_plain<T>(nxe, nye, kx, ky, 0, gpad, kf, gext, n_img, st))) return rc;
  fold_kernel<T><<<dim3((nx * ny + 255) / 256, n_img), 256, 0, st>>>(gext, nx, ny, cx, cy, gout);
  return check_launch("fold_kernel");
}

// log-likelihood and its gradient: the forward pipeline writes dlogL/dmodel,
// the adjoint of the PSF (a correlation with the kernel) gives dlogL/d(ray
// image) -- through the s x s mean's adjoint first when the convolution is
// supersampled -- and grad_kernel accumulates d(ray flux)/d(kwargs) per
// profile over the grid the convolution saw.
template <typename T>
int run_grad(const ModelArgs &m, const GridArgs &g, const lensim_psf *psf, int kx, int ky, int edge,
             const SSPlan &ss, const lensim_data *data, const double *params, int n_img, double *logl, double *grad,
             unsigned char *ws, const Layout &L, hipStream_t st) {
  T *gmodel = reinterpret_cast<T *>(ws + L.gmodel);
  const unsigned flags = LENSIM_IMAGE_SOURCE | LENSIM_IMAGE_LENS_LIGHT;
  MpKeep keep{};
  if (m.mp_n && m.n_source > 0) {
    const DeflGradPlan p = defl_grad_plan(m, size_t(g.nx) * g.ny * g.s * g.s, n_img);
    if (p.imgs >= n_img) {  // the store holds the whole batch
      keep.store = reinterpret_cast<double4 *>(ws + L.gstate);
      keep.per_img = p.per_img;
      keep.beta = ws + L.beta;
    }
  } else if (bulk_keeps<T>(m, size_t(g.nx) * g.ny * (ss.on ? size_t(ss.s) * ss.s : 1))) {
    keep.beta = ws + L.beta;
  }
  int d0, d1;
  const bool kept = sizeof(T) == sizeof(double) && L.gbeta && m.n_bulk == 0 && fast_model<T>(m, flags, d0, d1) &&
                    m.types[m.n_lens] == LENSIM_SERSIC_ELLIPSE;
  if (kept) keep.beta = ws + L.gbeta;
  int rc = ss.on ? run_image_ss<T>(m, g, psf, kx, ky, edge, ss, data, params, n_img, flags, nullptr, logl, ws, L, st,
                                   gmodel, keep)
                 : run_image<T>(m, g, psf, kx, ky, edge, data, params, n_img, flags, nullptr, logl, ws, L, st, gmodel, keep);
  if (rc) return rc;
  const bool identity = !psf || psf->type == LENSIM_PSF_NONE;
  const int kyp = kyp_of(ky);
  double *kf = reinterpret_cast<double *>(ws + L.psf);
  psf_prep_kernel<<<(kyp * kx + 255) / 256, 256, 0, st>>>(identity ? nullptr : psf->d_kernel, kx, ky, kyp, kf, 0);
  if ((rc = check_launch("psf_prep_kernel"))) return rc;
  T *glow = reinterpret_cast<T *>(ws + L.glow);
  T *gpad = reinterpret_cast<T *>(ws + L.gpad);
  T *gext = reinterpret_cast<T *>(ws + L.gext);
  const GridArgs gg = ss.on ? ray_grid(g) : g;  // the grid whose pixels the rays fill
  if (!ss.on) {
    if ((rc = adjoint_conv<T>(g.nx, g.ny, kx, ky, edge, gmodel, kf, glow, gpad, gext, n_img, st))) return rc;
  } else {
    T *gchr = reinterpret_cast<T *>(ws + L.gchr);
    const int nh = gg.nx * gg.ny;
    unpool_kernel<T><<<dim3((nh + 255) / 256, n_img), 256, 0, st>>>(gmodel, g.nx, g.ny, ss.s, 0, gchr);
    if ((rc = check_launch("unpool_kernel"))) return rc;
    if ((rc = adjoint_conv<T>(gg.nx, gg.ny, kx, ky, edge, gchr, kf, glow, gpad, gext, n_img, st))) return rc;
    if (ss.kxl > 0) {  // low-resolution part: adjoint of its convolution, then of the mean
      const int kypl = kyp_of(ss.kyl);
      double *kfl = reinterpret_cast<double *>(ws + L.psf_low);
      psf_prep_kernel<<<(kypl * ss.kxl + 255) / 256, 256, 0, st>>>(psf->d_kernel_low, ss.kxl, ss.kyl, kypl, kfl, 0);
      if ((rc = check_launch("psf_prep_kernel (low)"))) return rc;
      T *glu = reinterpret_cast<T *>(ws + L.glu);
      if ((rc = launch_conv_plain<T>(g.nx, g.ny, ss.kxl, ss.kyl, 0, gmodel, kfl, glu, n_img, st))) return rc;
      unpool_kernel<T><<<dim3((nh + 255) / 256, n_img), 256, 0, st>>>(glu, g.nx, g.ny, ss.s, 1, glow);
      if ((rc = check_launch("unpool_kernel"))) return rc;
    }
  }
  // per-profile gradients
  GradArgs ga;
  ga.params = params;
  ga.coefd = reinterpret_cast<const double *>(ws + L.coefd);
  ga.coeff = reinterpret_cast<const float *>(ws + L.coeff);
  ga.dcoefd = reinterpret_cast<const double *>(ws + L.dcoefd);
  ga.dcoeff = reinterpret_cast<const float *>(ws + L.dcoeff);
  ga.glow = glow;
  ga.gpart = reinterpret_cast<double *>(ws + L.gpart);
  ga.kept = kept;
  ga.gbeta = L.gbeta ? static_cast<void *>(ws + L.gbeta) : nullptr;
  ga.beta = L.beta ? static_cast<void *>(ws + L.beta) : nullptr;
  const int npix = gg.nx * gg.ny, nblk = (npix + 256 * kGradPix - 1) / (256 * kGradPix);
  const double *recd = reinterpret_cast<const double *>(ws + L.recd);
  const float *recf = reinterpret_cast<const float *>(ws + L.recf);
  // a multi-plane or bulk list first: it also stores beta (and dS/dbeta) at
  // every ray for the launches below
  if (m.mp_n || m.n_bulk > 0) {
    const int *tab = reinterpret_cast<const int *>(ws + L.mp_tab);
    double *gpart_mp = reinterpret_cast<double *>(ws + L.gpart_mp);
    double4 *store = reinterpret_cast<double4 *>(ws + L.gstate);
    rc = m.has_halo ? launch_defl_grad<T, true>(m, gg, ga, recd, recf, tab, gpart_mp, store, nblk, n_img, st)
                    : launch_defl_grad<T, false>(m, gg, ga, recd, recf, tab, gpart_mp, store, nblk, n_img, st);
    if (rc) return rc;
  }
  // then the sources: the first source's launch stores dS/dbeta at every ray
  // (ga.gbeta), which the inline lens launches after it read
  for (int q = 0; q < m.n_prof; ++q) {
    const int k = q < m.n_source ? m.n_defl + q : (q < m.n_source + m.n_defl ? q - m.n_source : q);
    if (m.mp_n && k < m.n_defl) continue;            // done above
    if (k >= m.n_lens && k < m.n_defl) continue;     // the bulk list, done above
    rc = m.has_halo ? launch_grad_profile<T, true>(m, gg, ga, recd, recf, nblk, n_img, k, st)
                    : launch_grad_profile<T, false>(m, gg, ga, recd, recf, nblk, n_img, k, st);
    if (rc) return rc;
  }
  const int n = n_img * m.n_prof * LENSIM_NPARAM;
  const DeflGradPlan pl = defl_grad_plan(m, size_t(gg.nx) * gg.ny * gg.s * gg.s, n_img);
  const int64_t rows = pl.n && pl.imgs >= n_img ? int64_t(n_img) * (m.n_defl - (m.mp_n ? 0 : m.n_lens)) : 0;
  const int list_blocks = int((rows + 3) / 4);
  grad_reduce_kernel<<<list_blocks + (n + 255) / 256, 256, 0, st>>>(
      m, reinterpret_cast<const int *>(ws + L.mp_tab), reinterpret_cast<const double *>(ws + L.gpart_mp), pl, list_blocks,
      n_img, ga.gpart, nblk, grad);
  return check_launch("grad_reduce_kernel");
}

// ------------------------------------------------- linear amplitude solve --
// ImageLinearFit.image_linear_solve (ImSim/image_linear_solve.py:98-181): the
// response of every linear light profile (its image at amp = 1,
// linear_response_matrix :362-455), weighted least squares against the data
// (de_lens.get_param_WLS, ImSim/de_lens.py:10-36) and the likelihood of the
// solved model (:229-340).
constexpr int kMaxLin = 8;  // linear amplitudes per model
constexpr int lin_acc(int n) { return n * (n + 1) / 2 + n; }  // M (upper triangle) and R

// Weights mask / C_D(data) (ImageModel.error_response, image_model.py:577-596:
// Data.C_D, the variance estimated from the data) and per-block partial sums
// of M = A W A^T (upper triangle) and R = A W d.  A is [N][n_img][npix].  N is
// fixed at compile time: the sums of eight amplitudes (44) cost two of them
// 22 us where their own five take 4.6 us (99^2, 16 images).
template <typename T, int N>
__global__ __launch_bounds__(256) void normal_kernel(ConvArgs c, const T *__restrict__ A, int n_img,
                                                     double *__restrict__ part) {
  constexpr int NA = lin_acc(N);
  const int img = blockIdx.y;
  const int npix = c.nx * c.ny;
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  double acc[NA];
#pragma unroll
  for (int q = 0; q < NA; ++q) acc[q] = 0.0;
  if (p < npix) {
    const size_t pd = p + size_t(img) * size_t(c.dstride);
    const double d = AT(c.data, pd);
    double var;
    if (c.noise) {
      var = AT(c.noise, pd) * AT(c.noise, pd);
    } else {
      const double t = c.expo ? AT(c.expo, p) : c.exposure_time;
      var = (d >= 0.0 ? d : 0.0) / t + c.bkg2;
    }
    const double w = (c.mask ? AT(c.mask, p) : 1.0) / var;
    double a[N];
#pragma unroll
    for (int l = 0; l < N; ++l) a[l] = double(AT(A, (size_t(l) * n_img + img) * npix + p));
    if (w != 0.0) {
      int q = 0;
#pragma unroll
      for (int i = 0; i < N; ++i) {
#pragma unroll
        for (int j = i; j < N; ++j) acc[q++] = a[i] * w * a[j];
      }
#pragma unroll
      for (int i = 0; i < N; ++i) acc[q++] = a[i] * w * d;
    }
  }
  __shared__ double red[4][NA];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int q = 0; q < NA; ++q) {
    const double v = wave_sum(acc[q]);
    if (lane == 0) red[wave][q] = v;
  }
  __syncthreads();
  if (threadIdx.x < NA) {
    const int q = threadIdx.x;
    AT(part, (size_t(img) * gridDim.x + blockIdx.x) * NA + q) = red[0][q] + red[1][q] + red[2][q] + red[3][q];
  }
}

// Eigenvalues of a symmetric N x N matrix (cyclic Jacobi rotations), in registers.
template <int N>
__device__ void sym_eigenvalues(double (&a)[N][N], double *ev) {
  for (int sweep = 0; sweep < 30; ++sweep) {
    double off = 0.0;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int j = i + 1; j < N; ++j) off += a[i][j] * a[i][j];
    if (off == 0.0) break;
#pragma unroll
    for (int p = 0; p < N; ++p)
#pragma unroll
      for (int q = p + 1; q < N; ++q) {
        if (a[p][q] == 0.0) continue;
        const double theta = (a[q][q] - a[p][p]) / (2.0 * a[p][q]);
        const double t = (theta >= 0.0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
        const double c = 1.0 / sqrt(t * t + 1.0), s = t * c;
#pragma unroll
        for (int k = 0; k < N; ++k) {  // columns p, q
          const double akp = a[k][p], akq = a[k][q];
          a[k][p] = c * akp - s * akq;
          a[k][q] = s * akp + c * akq;
        }
#pragma unroll
        for (int k = 0; k < N; ++k) {  // rows p, q
          const double apk = a[p][k], aqk = a[q][k];
          a[p][k] = c * apk - s * aqk;
          a[q][k] = s * apk + c * aqk;
        }
      }
  }
#pragma unroll
  for (int i = 0; i < N; ++i) ev[i] = a[i][i];
}

// LU factorisation with partial pivoting in place; returns the permutation
// parity (+1 / -1), 0 if a pivot is exactly zero.  The row exchanges are
// selections over the (compile-time) rows, so that the matrix stays in registers.
template <int N>
__device__ int lu_factor(double (&a)[N][N], int (&piv)[N]) {
  int parity = 1;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    int pr = k;
    double best = fabs(a[k][k]);
#pragma unroll
    for (int i = k + 1; i < N; ++i)
      if (fabs(a[i][k]) > best) {
        best = fabs(a[i][k]);
        pr = i;
      }
    piv[k] = pr;
    if (pr != k) parity = -parity;
#pragma unroll
    for (int i = k + 1; i < N; ++i)
      if (pr == i) {
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const double t = a[k][j];
          a[k][j] = a[i][j];
          a[i][j] = t;
        }
      }
    if (a[k][k] == 0.0) return 0;
#pragma unroll
    for (int i = k + 1; i < N; ++i) {
      a[i][k] /= a[k][k];
#pragma unroll
      for (int j = k + 1; j < N; ++j) a[i][j] -= a[i][k] * a[k][j];
    }
  }
  return parity;
}

template <int N>
__device__ void lu_solve(const double (&lu)[N][N], const int (&piv)[N], double (&b)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k) {
#pragma unroll
    for (int i = k + 1; i < N; ++i)
      if (piv[k] == i) {
        const double t = b[k];
        b[k] = b[i];
        b[i] = t;
      }
  }
#pragma unroll
  for (int i = 1; i < N; ++i)
#pragma unroll
    for (int j = 0; j < i; ++j) b[i] -= lu[i][j] * b[j];
#pragma unroll
  for (int i = N - 1; i >= 0; --i) {
#pragma unroll
    for (int j = i + 1; j < N; ++j) b[i] -= lu[i][j] * b[j];
    b[i] /= lu[i][i];
  }
}

// One wave per image: its lanes sum the partials (lane l blocks l, l + 64, ...,
// then the fixed wave sum), then every lane checks cond(M) < 5 / eps, solves
// M B = R (B = 0 when unstable or not finite), optionally inverts M
// (nan_to_num'ed, zero when unstable) and the marginalisation constant
// (de_lens.marginalisation_const / marginalization_new, de_lens.py:40-77) in
// registers, and the first stores.  One thread per image with its matrices in
// scratch memory and 44 serial sums took 171 us for 16 images, this 11.
template <int N>
__global__ __launch_bounds__(64) void lin_solve_kernel(const double *__restrict__ part, int nblk, int source_marg,
                                                       double d_prior, double *__restrict__ amp,
                                                       double *__restrict__ amp_out, double *__restrict__ cov,
                                                       double *__restrict__ marg) {
  constexpr int NA = lin_acc(N);
  const int img = blockIdx.x, lane = threadIdx.x;
  double acc[NA];
#pragma unroll
  for (int q = 0; q < NA; ++q) acc[q] = 0.0;
  for (int b = lane; b < nblk; b += 64)
#pragma unroll
    for (int q = 0; q < NA; ++q) acc[q] += AT(part, (size_t(img) * nblk + b) * NA + q);
#pragma unroll
  for (int q = 0; q < NA; ++q) acc[q] = wave_sum(acc[q]);
  double M[N][N], W[N][N], B[N];
  {
    int q = 0;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int j = i; j < N; ++j) M[i][j] = M[j][i] = acc[q++];
#pragma unroll
    for (int i = 0; i < N; ++i) B[i] = acc[q++];
  }
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int j = 0; j < N; ++j) W[i][j] = M[i][j];
  double ev[N];
  sym_eigenvalues<N>(W, ev);
  double emax = 0.0, emin = INFINITY;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    emax = fmax(emax, fabs(ev[i]));
    emin = fmin(emin, fabs(ev[i]));
  }
  const double eps = 2.220446049250313e-16;
  const bool stable = emin > 0.0 && emax / emin < 5.0 / eps;
  int piv[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    piv[i] = i;
#pragma unroll
    for (int j = 0; j < N; ++j) W[i][j] = M[i][j];
  }
  const int parity = lu_factor<N>(W, piv);
  const bool ok = stable && parity != 0;
  bool finite = ok;
  if (finite) {
    lu_solve<N>(W, piv, B);
#pragma unroll
    for (int i = 0; i < N; ++i) finite = finite && isfinite(B[i]);
  }
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (lane == 0) {
      const double v = finite ? B[i] : 0.0;
      AT(amp, size_t(img) * N + i) = v;
      if (amp_out) AT(amp_out, size_t(img) * N + i) = v;
    }
  if (cov) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      double e[N];
#pragma unroll
      for (int i = 0; i < N; ++i) e[i] = i == j ? 1.0 : 0.0;
      if (ok) lu_solve<N>(W, piv, e);
#pragma unroll
      for (int i = 0; i < N; ++i)
        if (lane == 0) AT(cov, (size_t(img) * N + i) * N + j) = (ok && isfinite(e[i])) ? e[i] : 0.0;
    }
  }
  double mc = 0.0;
  if (source_marg) {
    if (!ok) {
      mc = -1e15;  // slogdet / eig of a zero covariance
    } else if (!(d_prior > 0.0)) {
      // 1/2 log det(M^-1) = -1/2 sum log|U_ii| with the sign of det(M)
      double logdet = 0.0;
      int sign = parity;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        logdet += log(fabs(W[i][i]));
        if (W[i][i] < 0.0) sign = -sign;
      }
      mc = sign * (-logdet) / 2.0;
    } else {
      // eigenvalues of M^-1 = 1 / eigenvalues of M, clipped at d_prior^2
      double ld = 0.0, sgn = 1.0;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const double v = 1.0 / ev[i];
        sgn *= v > 0.0 ? 1.0 : (v < 0.0 ? -1.0 : 0.0);
        ld += log(fmin(fabs(v), d_prior * d_prior));
      }
      const double log_det = ld * sgn;
      mc = isnan(log_det) ? -1e15 : log_det / 2.0 + N / 2.0 * log(M_PI / 2.0) - N * log(d_prior);
    }
  }
  if (lane == 0) AT(marg, img) = mc;
}

// normal_kernel and lin_solve_kernel for n_lin amplitudes (1 .. kMaxLin).
template <typename T, int N = kMaxLin>
int launch_normal_solve(const ConvArgs &c, const T *A, int n_lin, int n_img, int nblk, double *part, int source_marg,
                        double d_prior, double *amp, double *amp_out, double *cov, double *marg, hipStream_t st) {
  if constexpr (N > 1) {
    if (n_lin < N)
      return launch_normal_solve<T, N - 1>(c, A, n_lin, n_img, nblk, part, source_marg, d_prior, amp, amp_out, cov, marg,
                                           st);
  }
  normal_kernel<T, N><<<dim3(nblk, n_img), 256, 0, st>>>(c, A, n_img, part);
  int rc = check_launch("normal_kernel");
  if (rc) return rc;
  lin_solve_kernel<N><<<n_img, 64, 0, st>>>(part, nblk, source_marg, d_prior, amp, amp_out, cov, marg);
  return check_launch("lin_solve_kernel");
}

// Solved model (zero outside the likelihood mask, array_masked2image) and its chi^2.
template <typename T>
__global__ __launch_bounds__(256) void lin_model_kernel(ConvArgs c, const T *__restrict__ A, const double *__restrict__ amp,
                                                        int n_lin, int n_img, T *__restrict__ out,
                                                        double *__restrict__ partial) {
  const int img = blockIdx.y;
  const int npix = c.nx * c.ny;
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  double chi = 0.0;
  if (p < npix) {
    double m = 0.0;
    if (!c.mask || AT(c.mask, p) != 0.0)
      for (int l = 0; l < n_lin; ++l)
        m += AT(amp, size_t(img) * n_lin + l) * double(AT(A, (size_t(l) * n_img + img) * npix + p));
    const T mt = T(m);
    if (out) AT(out, size_t(img) * npix + p) = mt;
    chi = chi2_pixel<T>(c, p, mt, img);
  }
  __shared__ double red[4];
  for (int off = 32; off > 0; off >>= 1) chi += __shfl_xor(chi, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = chi;
  __syncthreads();
  if (threadIdx.x == 0) AT(partial, size_t(img) * gridDim.x + blockIdx.x) = red[0] + red[1] + red[2] + red[3];
}

// Workspace of the linear solve: the image layout of one column, the columns A
// with their pooled images and block maxima (all columns are convolved in one
// launch), partials, amplitudes and constants.
struct LinLayout {
  Layout img;
  size_t A, low, blkmax, part, chi, amp, marg, total;
};

LinLayout lin_layout(const ModelArgs &m, int nx, int ny, int kx, int ky, int n_img, int precision, const SSPlan &ss,
                     int n_lin) {
  LinLayout L;
  L.img = layout(m, nx, ny, kx, ky, n_img, precision, ss);
  const size_t tsz = precision == LENSIM_MIXED ? 4 : 8;
  const size_t npix = size_t(nx) * ny, nblk = (npix + 255) / 256;
  size_t off = L.img.total;
  L.A = off;
  off = align256(off + size_t(n_lin) * n_img * npix * tsz);
  L.low = L.blkmax = off;
  if (!ss.on) {
    off = align256(off + size_t(n_lin) * n_img * npix * tsz);
    L.blkmax = off;
    off = align256(off + size_t(n_lin) * n_img * nblk * 4);
  }
  L.part = off;
  off = align256(off + size_t(n_img) * nblk * lin_acc(n_lin) * 8);
  L.chi = off;
  off = align256(off + size_t(n_img) * nblk * 8);
  L.amp = off;
  off = align256(off + size_t(n_img) * kMaxLin * 8);
  L.marg = off;
  off = align256(off + size_t(n_img) * 8);
  L.total = off;
  return L;
}

// The response columns of run_linear without supersampled convolution: the
// records (at amp = 1) and the PSF prepared once, a render per light profile
// (every other one left out), one convolution over all columns' images.
template <typename T>
int run_responses(const ModelArgs &m_in, const GridArgs &g, const lensim_psf *psf, int kx, int ky, int edge,
                  const double *params, int n_img, int n_lin, T *A, unsigned char *ws, const LinLayout &LL,
                  hipStream_t st) {
  const Layout &L = LL.img;
  ModelArgs m = with_grid(m_in, g);
  const ConvChoice<T> cc(psf, 0, kx, ky, ws, L);
  int rc = launch_prep_psf(m, params, n_img, cc.job, false, ws, L, st);
  if (rc) return rc;
  const size_t npix = size_t(g.nx) * g.ny, nblk = (npix + 255) / 256;
  T *low = reinterpret_cast<T *>(ws + LL.low);
  float *blkmax = cc.mfma ? reinterpret_cast<float *>(ws + LL.blkmax) : nullptr;
  for (int l = 0; l < n_lin; ++l) {
    ModelArgs mc = m;
    for (int k = 0; k < n_lin; ++k)
      if (k != l) mc.types[m.n_lens + k] = LENSIM_NULL;
    rc = launch_render<T>(mc, g, reinterpret_cast<const double *>(ws + L.recd),
                          reinterpret_cast<const float *>(ws + L.recf),
                          reinterpret_cast<const double *>(ws + L.coefd),
                          reinterpret_cast<const float *>(ws + L.coeff), reinterpret_cast<const int *>(ws + L.mp_tab),
                          l < m.n_source ? LENSIM_IMAGE_SOURCE : LENSIM_IMAGE_LENS_LIGHT, MpKeep{},
                          low + size_t(l) * n_img * npix, blkmax ? blkmax + size_t(l) * n_img * nblk : nullptr, n_img,
                          st);
    if (rc) return rc;
  }
  ConvArgs c{};
  c.nx = g.nx;
  c.ny = g.ny;
  c.kx = kx;
  c.ky = ky;
  c.kyp = cc.job.kyp;
  c.edge = edge;
  const int all = n_img * n_lin, most = 65535;  // images a launch's grid holds
  for (int i = 0; i < all; i += most) {
    int n_tiles;
    rc = launch_conv<T>(c, cc, all - i < most ? all - i : most, low + i * npix, blkmax ? blkmax + i * nblk : nullptr,
                        A + i * npix, nullptr, &n_tiles, st);
    if (rc) return rc;
  }
  return LENSIM_OK;
}

template <typename T>
int run_linear(const ModelArgs &m_in, const GridArgs &g, const lensim_psf *psf, int kx, int ky, int edge,
               const SSPlan &ss, const lensim_data *data, const double *params, int n_img, int source_marg,
               double d_prior, double *amp_out, double *logl, T *model_out, double *cov, T *resp_out,
               unsigned char *ws, const LinLayout &LL, hipStream_t st) {
  ModelArgs m = m_in;
  m.unit_amp = 1;
  const int n_lin = m.n_source + m.n_light;
  const int npix = g.nx * g.ny, nblk = (npix + 255) / 256;
  T *A = resp_out ? resp_out : reinterpret_cast<T *>(ws + LL.A);
  int rc = LENSIM_OK;
  if (!ss.on) {
    if ((rc = run_responses<T>(m, g, psf, kx, ky, edge, params, n_img, n_lin, A, ws, LL, st))) return rc;
  } else {
    // one column per linear profile: the model with every other light profile off
    for (int l = 0; l < n_lin; ++l) {
      ModelArgs mc = m;
      for (int k = m.n_lens; k < m.n_lens + n_lin; ++k)
        if (k - m.n_lens != l) mc.types[k] = LENSIM_NULL;
      const unsigned flags = l < m.n_source ? LENSIM_IMAGE_SOURCE : LENSIM_IMAGE_LENS_LIGHT;
      rc = run_image_ss<T>(mc, g, psf, kx, ky, edge, ss, nullptr, params, n_img, flags, A + size_t(l) * n_img * npix,
                           nullptr, ws, LL.img, st);
      if (rc) return rc;
    }
  }
  ConvArgs c{};
  c.nx = g.nx;
  c.ny = g.ny;
  c.data = data->d_data;
  c.noise = data->d_noise_map;
  c.expo = data->d_exposure_map;
  c.mask = data->d_mask;
  c.exposure_time = data->exposure_time;
  c.bkg2 = data->background_rms * data->background_rms;
  c.inv_t = 1.0 / data->exposure_time;
  c.dstride = data->image_stride;
  double *amp = reinterpret_cast<double *>(ws + LL.amp);
  double *marg = reinterpret_cast<double *>(ws + LL.marg);
  rc = launch_normal_solve<T>(c, A, n_lin, n_img, nblk, reinterpret_cast<double *>(ws + LL.part), source_marg, d_prior,
                              amp, amp_out, cov, marg, st);
  if (rc) return rc;
  double *chi = reinterpret_cast<double *>(ws + LL.chi);
  lin_model_kernel<T><<<dim3(nblk, n_img), 256, 0, st>>>(c, A, amp, n_lin, n_img, model_out, chi);
  if ((rc = check_launch("lin_model_kernel"))) return rc;
  logl_kernel<<<n_img, 64, 0, st>>>(chi, nblk, marg, logl);
  return check_launch("logl_kernel");
}

// ------------------------------------------- allocation-free entry point --
// lensim_loglike_noalloc keeps its scratch memory in this file-scope device
// array (one copy per GPU, held until the process ends) instead of a
// workspace argument.  In host code `scratch` names a host-side stand-in, not
// the device array: its device address on the current GPU comes from
// hipGetSymbolAddress (scratch_on_device) and only that address reaches
// kernels.  No kernel of the log-likelihood pipeline reads scratch memory it
// has not written earlier in the same call, so nothing is cleared between
// calls.  Calls that overlap on one GPU share the array and race.
constexpr size_t kScratchBytes = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};

// The device address of `scratch` on the current GPU, looked up once per GPU.
int scratch_on_device(void **out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  if (dev < 0 || dev >= kMaxDevices) return fail(LENSIM_EINVAL, "device %d beyond the %d supported", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
    if (!p) return fail(LENSIM_EDEVICE, "hipGetSymbolAddress(scratch) returned NULL");
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return LENSIM_OK;
}

int check_ws(const Layout &L, void *ws, size_t ws_bytes) {
  if (L.total > ws_bytes)
    return fail(LENSIM_EWORKSPACE, "workspace of %zu B is smaller than the %zu B needed", ws_bytes, L.total);
  if (L.total > 0 && !ws) return fail(LENSIM_EINVAL, "workspace pointer is NULL");
  if (reinterpret_cast<uintptr_t>(ws) & 255) return fail(LENSIM_EINVAL, "workspace must be 256-byte aligned");
  return LENSIM_OK;
}

// The caller's buffers that a call reads: parameters, the bulk type list, the
// multi-plane arrays, the evaluation mask, the PSF kernels and the data, each
// with the extent the header gives it.
void add_inputs(CallRanges &cr, const lensim_model *model, const ModelArgs &m, const double *params, int n_img,
                const lensim_grid *grid, const lensim_psf *psf, const lensim_data *data, int nx, int ny) {
  cr.add(params, size_t(n_img) * m.n_prof * LENSIM_NPARAM * sizeof(double));
  if (m.bulk_types) cr.add(m.bulk_types, size_t(m.n_bulk) * sizeof(int32_t));
  if (const lensim_multiplane *mp = model->multiplane) {
    const size_t n = mp->stride ? size_t(n_img - 1) * size_t(mp->stride) + mp->n_planes : size_t(mp->n_planes);
    cr.add(mp->d_order, size_t(mp->n_planes - 1) * sizeof(int32_t));
    cr.add(mp->d_T_ij, n * sizeof(double));
    cr.add(mp->d_T_z, n * sizeof(double));
    cr.add(mp->d_r2p, n * sizeof(double));
  }
  if (grid) cr.add(grid->d_eval_mask, size_t(grid->nx) * grid->ny);
  if (psf) {
    cr.add(psf->d_kernel, size_t(psf->kx) * psf->ky * sizeof(double));
    cr.add(psf->d_kernel_low, size_t(psf->kx_low) * psf->ky_low * sizeof(double));
  }
  if (data) {
    const size_t npix = size_t(nx) * ny;
    const size_t nd = data->image_stride ? size_t(n_img - 1) * size_t(data->image_stride) + npix : npix;
    cr.add(data->d_data, nd * sizeof(double));
    cr.add(data->d_noise_map, nd * sizeof(double));
    cr.add(data->d_exposure_map, npix * sizeof(double));
    cr.add(data->d_mask, npix * sizeof(double));
  }
}

#ifdef LENSIM_BOUNDS_CHECK
// Stores bytes 0 .. n - 1 of buf and then byte n (one past the registered range).
__global__ void bounds_selftest_kernel(unsigned char *buf, size_t n) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i <= n) AT(buf, i) = static_cast<unsigned char>(i & 255);
}
#endif

}  // namespace

// ------------------------------------------------------------- C ABI -----

extern "C" {

int lensim_abi_version(void) { return LENSIM_ABI_VERSION; }

int lensim_timing_enable(int on) {
  g_timing = on != 0;
  return LENSIM_OK;
}

int lensim_timing_read(double *render_ms, double *conv_ms, int64_t *calls) {
  double r = 0.0, c = 0.0;
  int64_t n = 0;
  for (int i = 0; i < g_ncalls; ++i) {
    TimedCall &tc = g_calls[i];
    if (!tc.ev[0] || !tc.ev[1] || !tc.ev[2]) continue;
    hipError_t e = hipEventSynchronize(tc.ev[2]);
    if (e != hipSuccess) return hip_fail(e, "hipEventSynchronize");
    float a = 0.f, b = 0.f;
    if (hipEventElapsedTime(&a, tc.ev[0], tc.ev[1]) != hipSuccess ||
        hipEventElapsedTime(&b, tc.ev[1], tc.ev[2]) != hipSuccess)
      return fail(LENSIM_EDEVICE, "hipEventElapsedTime failed");
    r += a;
    c += b;
    ++n;
  }
  g_ncalls = 0;  // events are kept and reused by later calls
  if (render_ms) *render_ms = r;
  if (conv_ms) *conv_ms = c;
  if (calls) *calls = n;
  return LENSIM_OK;
}

const char *lensim_last_error(void) { return g_err; }

int lensim_bounds_checked(void) {
#ifdef LENSIM_BOUNDS_CHECK
  return 1;
#else
  return 0;
#endif
}

int lensim_bounds_selftest(void *d_buf, size_t bytes, void *stream) {
#ifdef LENSIM_BOUNDS_CHECK
  if (!d_buf) return fail(LENSIM_EINVAL, "NULL buffer");
  if (bytes == 0 || bytes > (size_t(1) << 20)) return fail(LENSIM_EINVAL, "bytes must be in [1, 2^20]");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  CallRanges cr;
  cr.add(d_buf, bytes);
  int rc = cr.begin(st);
  if (rc) return rc;
  bounds_selftest_kernel<<<unsigned((bytes + 1 + 255) / 256), 256, 0, st>>>(static_cast<unsigned char *>(d_buf),
                                                                             bytes);
  return cr.end(st, check_launch("bounds_selftest_kernel"));
#else
  (void)d_buf;
  (void)bytes;
  (void)stream;
  return fail(LENSIM_EUNSUPPORTED, "lensim_bounds_selftest needs the bounds-checked build (liblensim_checked.so)");
#endif
}

size_t lensim_workspace_size(const lensim_model *model, const lensim_grid *grid, const lensim_psf *psf,
                             int32_t n_img, int32_t precision) {
  ModelArgs m;
  if (model_args(model, m)) return 0;
  int nx = 1, ny = 1;
  SSPlan ss;
  if (grid) {
    nx = grid->nx;
    ny = grid->ny;
    GridArgs g;
    if (grid_args(grid, g) || psf_ss(psf, g, 0, ss)) return 0;
  }
  int kx = 1, ky = 1, edge = 0;
  if (psf_dims(psf, 0, kx, ky, edge)) return 0;
  return layout(m, nx, ny, kx, ky, n_img, precision, ss).total;
}

int lensim_raytrace(const lensim_model *model, const double *d_params, int32_t n_img, const double *d_x,
                    const double *d_y, int64_t n_ray, int32_t precision, double *d_beta_x, double *d_beta_y,
                    void *ws, size_t ws_bytes, void *stream) {
  ModelArgs m;
  int rc = model_args(model, m);
  if (rc) return rc;
  if (n_img < 0 || n_ray < 0) return fail(LENSIM_EINVAL, "negative sizes");
  if (n_img == 0 || n_ray == 0) return LENSIM_OK;
  if (n_ray > (int64_t(1) << 36)) return fail(LENSIM_EINVAL, "n_ray too large");
  if (n_img > 65535) return fail(LENSIM_EINVAL, "n_img %d exceeds 65535 per call", n_img);
  if (!d_x || !d_y || !d_beta_x || !d_beta_y || (m.n_prof && !d_params))
    return fail(LENSIM_EINVAL, "NULL buffer");
  if (precision != LENSIM_FP64 && precision != LENSIM_MIXED) return fail(LENSIM_EINVAL, "bad precision");
  const Layout L = layout(m, 1, 1, 1, 1, n_img, precision);
  if ((rc = check_ws(L, ws, ws_bytes))) return rc;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  unsigned char *w = static_cast<unsigned char *>(ws);
  CallRanges cr;
  add_inputs(cr, model, m, d_params, n_img, nullptr, nullptr, nullptr, 0, 0);
  cr.add(d_x, size_t(n_ray) * sizeof(double));
  cr.add(d_y, size_t(n_ray) * sizeof(double));
  cr.add(d_beta_x, size_t(n_img) * size_t(n_ray) * sizeof(double));
  cr.add(d_beta_y, size_t(n_img) * size_t(n_ray) * sizeof(double));
  cr.add(ws, L.total);
  if ((rc = cr.begin(st))) return rc;
  const bool runs_in_prep = m.mp_n > 0 && m.mp_n <= kMpPrep;
  rc = runs_in_prep ? launch_prep_psf(m, d_params, n_img, PsfJob{}, false, w, L, st)
                    : launch_prep(m, d_params, n_img, w, L, st);
  if (rc) return cr.end(st, rc);
  dim3 grid((unsigned)((n_ray + 255) / 256), n_img);
  const double *recd = reinterpret_cast<const double *>(w + L.recd);
  const float *recf = reinterpret_cast<const float *>(w + L.recf);
  const double *coefd = reinterpret_cast<const double *>(w + L.coefd);
  const float *coeff = reinterpret_cast<const float *>(w + L.coeff);
  if (m.mp_n) {
    int *tab = reinterpret_cast<int *>(w + L.mp_tab);
    if (!runs_in_prep && (rc = launch_mp_runs(m, tab, n_img, st))) return cr.end(st, rc);
    rc = precision == LENSIM_FP64 ? launch_raytrace_mp<double>(m, recd, recf, coefd, coeff, tab, d_x, d_y, n_ray, n_img,
                                                               d_beta_x, d_beta_y, st)
                                  : launch_raytrace_mp<float>(m, recd, recf, coefd, coeff, tab, d_x, d_y, n_ray, n_img,
                                                              d_beta_x, d_beta_y, st);
    return cr.end(st, rc);
  }
#define LENSIM_TRACE(T, H, D)                                                                                     \
  raytrace_kernel<T, H, D><<<grid, 256, 0, st>>>(m, recd, recf, coefd, coeff, d_x, d_y, n_ray, d_beta_x, d_beta_y)
  if (precision == LENSIM_FP64) {
    if (m.has_halo) LENSIM_TRACE(double, true, false);
    else LENSIM_TRACE(double, false, false);
  } else if (m.has_nie_nfw) {  // SIE / NIE and NFW deflect in double (see nie_defl)
    if (m.has_halo) LENSIM_TRACE(float, true, true);
    else LENSIM_TRACE(float, false, true);
  } else {
    if (m.has_halo) LENSIM_TRACE(float, true, false);
    else LENSIM_TRACE(float, false, false);
  }
#undef LENSIM_TRACE
  return cr.end(st, check_launch("raytrace_kernel"));
}

int lensim_surface_brightness(const lensim_model *model, const double *d_params, int32_t n_img, int32_t which,
                              const double *d_x, const double *d_y, int64_t n_ray, int32_t precision,
                              double *d_flux, void *ws, size_t ws_bytes, void *stream) {
  ModelArgs m;
  int rc = model_args(model, m);
  if (rc) return rc;
  if (n_img < 0 || n_ray < 0) return fail(LENSIM_EINVAL, "negative sizes");
  if (which != 0 && which != 1) return fail(LENSIM_EINVAL, "which must be 0 (source) or 1 (lens light)");
  if (n_img == 0 || n_ray == 0) return LENSIM_OK;
  if (n_ray > (int64_t(1) << 36)) return fail(LENSIM_EINVAL, "n_ray too large");
  if (n_img > 65535) return fail(LENSIM_EINVAL, "n_img %d exceeds 65535 per call", n_img);
  if (!d_x || !d_y || !d_flux || (m.n_prof && !d_params)) return fail(LENSIM_EINVAL, "NULL buffer");
  if (precision != LENSIM_FP64 && precision != LENSIM_MIXED) return fail(LENSIM_EINVAL, "bad precision");
  const Layout L = layout(m, 1, 1, 1, 1, n_img, precision);
  if ((rc = check_ws(L, ws, ws_bytes))) return rc;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  unsigned char *w = static_cast<unsigned char *>(ws);
  CallRanges cr;
  add_inputs(cr, model, m, d_params, n_img, nullptr, nullptr, nullptr, 0, 0);
  cr.add(d_x, size_t(n_ray) * sizeof(double));
  cr.add(d_y, size_t(n_ray) * sizeof(double));
  cr.add(d_flux, size_t(n_img) * size_t(n_ray) * sizeof(double));
  cr.add(ws, L.total);
  if ((rc = cr.begin(st))) return rc;
  if ((rc = launch_prep(m, d_params, n_img, w, L, st))) return cr.end(st, rc);
  const int k0 = which == 0 ? m.n_defl : m.n_defl + m.n_source;
  const int k1 = which == 0 ? m.n_defl + m.n_source : m.n_prof;
  dim3 grid((unsigned)((n_ray + 255) / 256), n_img);
  if (precision == LENSIM_FP64)
    light_kernel<double><<<grid, 256, 0, st>>>(m, reinterpret_cast<double *>(w + L.recd),
                                                reinterpret_cast<float *>(w + L.recf), k0, k1, d_x, d_y, n_ray,
                                                d_flux);
  else
    light_kernel<float><<<grid, 256, 0, st>>>(m, reinterpret_cast<double *>(w + L.recd),
                                               reinterpret_cast<float *>(w + L.recf), k0, k1, d_x, d_y, n_ray,
                                               d_flux);
  return cr.end(st, check_launch("light_kernel"));
}

int lensim_image(const lensim_model *model, const lensim_grid *grid, const lensim_psf *psf, const double *d_params,
                 int32_t n_img, int32_t precision, uint32_t flags, void *d_out, void *ws, size_t ws_bytes,
                 void *stream) {
  ModelArgs m;
  int rc = model_args(model, m);
  if (rc) return rc;
  GridArgs g;
  if ((rc = grid_args(grid, g))) return rc;
  int kx, ky, edge;
  if ((rc = psf_dims(psf, flags, kx, ky, edge))) return rc;
  if (n_img < 0) return fail(LENSIM_EINVAL, "negative n_img");
  if (n_img == 0) return LENSIM_OK;
  if (n_img > 65535) return fail(LENSIM_EINVAL, "n_img %d exceeds 65535 per call", n_img);
  if (!d_out || (m.n_prof && !d_params)) return fail(LENSIM_EINVAL, "NULL buffer");
  if (precision != LENSIM_FP64 && precision != LENSIM_MIXED) return fail(LENSIM_EINVAL, "bad precision");
  // kernel dims used by the layout: the real PSF unless unconvolved
  int lkx = 1, lky = 1, le = 0;
  psf_dims(psf, 0, lkx, lky, le);
  SSPlan ss, ss_layout;
  if ((rc = psf_ss(psf, g, flags, ss))) return rc;
  if ((rc = psf_ss(psf, g, 0, ss_layout))) return rc;
  const Layout L = layout(m, g.nx, g.ny, lkx, lky, n_img, precision, ss_layout);
  if ((rc = check_ws(L, ws, ws_bytes))) return rc;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  unsigned char *w = static_cast<unsigned char *>(ws);
  const size_t tsz = precision == LENSIM_FP64 ? sizeof(double) : sizeof(float);
  CallRanges cr;
  add_inputs(cr, model, m, d_params, n_img, grid, psf, nullptr, g.nx, g.ny);
  cr.add(d_out, size_t(n_img) * g.nx * g.ny * tsz);
  cr.add(ws, L.total);
  if ((rc = cr.begin(st))) return rc;
  if (ss.on) {
    if (precision == LENSIM_FP64)
      rc = run_image_ss<double>(m, g, psf, kx, ky, edge, ss, nullptr, d_params, n_img, flags,
                                static_cast<double *>(d_out), nullptr, w, L, st);
    else
      rc = run_image_ss<float>(m, g, psf, kx, ky, edge, ss, nullptr, d_params, n_img, flags,
                               static_cast<float *>(d_out), nullptr, w, L, st);
  } else if (precision == LENSIM_FP64) {
    rc = run_image<double>(m, g, psf, kx, ky, edge, nullptr, d_params, n_img, flags, static_cast<double *>(d_out),
                           nullptr, w, L, st);
  } else {
    rc = run_image<float>(m, g, psf, kx, ky, edge, nullptr, d_params, n_img, flags, static_cast<float *>(d_out),
                          nullptr, w, L, st);
  }
  return cr.end(st, rc);
}

int lensim_loglike(const lensim_model *model, const lensim_grid *grid, const lensim_psf *psf,
                   const lensim_data *data, const double *d_params, int32_t n_img, int32_t precision,
                   double *d_logl, void *d_model_out, void *ws, size_t ws_bytes, void *stream) {
  ModelArgs m;
  int rc = model_args(model, m);
  if (rc) return rc;
  GridArgs g;
  if ((rc = grid_args(grid, g))) return rc;
  int kx, ky, edge;
  if ((rc = psf_dims(psf, 0, kx, ky, edge))) return rc;
  if (!data || !data->d_data) return fail(LENSIM_EINVAL, "data image is NULL");
  if (!data->d_noise_map && !data->d_exposure_map && !(data->exposure_time > 0.0))
    return fail(LENSIM_EINVAL, "need a noise map, an exposure map or a positive exposure time");
  if (data->image_stride != 0 && data->image_stride < int64_t(g.nx) * g.ny)
    return fail(LENSIM_EINVAL, "image_stride %lld is smaller than an image", (long long)data->image_stride);
  if (n_img < 0) return fail(LENSIM_EINVAL, "negative n_img");
  if (n_img == 0) return LENSIM_OK;
  if (n_img > 65535) return fail(LENSIM_EINVAL, "n_img %d exceeds 65535 per call", n_img);
  if (!d_logl || (m.n_prof && !d_params)) return fail(LENSIM_EINVAL, "NULL buffer");
  if (precision != LENSIM_FP64 && precision != LENSIM_MIXED) return fail(LENSIM_EINVAL, "bad precision");
  SSPlan ss;
  if ((rc = psf_ss(psf, g, 0, ss))) return rc;
  const Layout L = layout(m, g.nx, g.ny, kx, ky, n_img, precision, ss);
  if ((rc = check_ws(L, ws, ws_bytes))) return rc;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  unsigned char *w = static_cast<unsigned char *>(ws);
  const unsigned flags = LENSIM_IMAGE_SOURCE | LENSIM_IMAGE_LENS_LIGHT;
  const size_t tsz = precision == LENSIM_FP64 ? sizeof(double) : sizeof(float);
  CallRanges cr;
  add_inputs(cr, model, m, d_params, n_img, grid, psf, data, g.nx, g.ny);
  cr.add(d_logl, size_t(n_img) * sizeof(double));
  cr.add(d_model_out, size_t(n_img) * g.nx * g.ny * tsz);
  cr.add(ws, L.total);
  if ((rc = cr.begin(st))) return rc;
  if (ss.on) {
    if (precision == LENSIM_FP64)
      rc = run_image_ss<double>(m, g, psf, kx, ky, edge, ss, data, d_params, n_img, flags,
                                static_cast<double *>(d_model_out), d_logl, w, L, st);
    else
      rc = run_image_ss<float>(m, g, psf, kx, ky, edge, ss, data, d_params, n_img, flags,
                               static_cast<float *>(d_model_out), d_logl, w, L, st);
  } else if (precision == LENSIM_FP64) {
    rc = run_image<double>(m, g, psf, kx, ky, edge, data, d_params, n_img, flags, static_cast<double *>(d_model_out),
                           d_logl, w, L, st);
  } else {
    rc = run_image<float>(m, g, psf, kx, ky, edge, data, d_params, n_img, flags, static_cast<float *>(d_model_out),
                          d_logl, w, L, st);
  }
  return cr.end(st, rc);
}

size_t lensim_data_loglike_workspace_size(int32_t nx, int32_t ny, int32_t n_img) {
  if (nx <= 0 || ny <= 0 || n_img < 0) return 0;
  return align256(size_t(n_img) * ((size_t(nx) * ny + 255) / 256) * 8) + 256;
}

int lensim_data_loglike(const lensim_data *data, int32_t nx, int32_t ny, const void *d_model, int32_t n_img,
                        int32_t precision, double *d_logl, void *ws, size_t ws_bytes, void *stream) {
  if (nx <= 0 || ny <= 0) return fail(LENSIM_EINVAL, "image sizes must be positive (nx=%d ny=%d)", nx, ny);
  if (int64_t(nx) * ny > (int64_t(1) << 30)) return fail(LENSIM_EINVAL, "image too large");
  if (!data || !data->d_data) return fail(LENSIM_EINVAL, "data image is NULL");
  if (!data->d_noise_map && !data->d_exposure_map && !(data->exposure_time > 0.0))
    return fail(LENSIM_EINVAL, "need a noise map, an exposure map or a positive exposure time");
  if (data->image_stride != 0 && data->image_stride < int64_t(nx) * ny)
    return fail(LENSIM_EINVAL, "image_stride %lld is smaller than an image", (long long)data->image_stride);
  if (n_img < 0) return fail(LENSIM_EINVAL, "negative n_img");
  if (n_img == 0) return LENSIM_OK;
  if (n_img > 65535) return fail(LENSIM_EINVAL, "n_img %d exceeds 65535 per call", n_img);
  if (!d_model || !d_logl) return fail(LENSIM_EINVAL, "NULL buffer");
  if (precision != LENSIM_FP64 && precision != LENSIM_MIXED) return fail(LENSIM_EINVAL, "bad precision");
  const size_t need = lensim_data_loglike_workspace_size(nx, ny, n_img);
  if (ws_bytes < need) return fail(LENSIM_EWORKSPACE, "workspace of %zu B is smaller than the %zu B needed", ws_bytes,
                                   need);
  if (!ws || (reinterpret_cast<uintptr_t>(ws) & 255)) return fail(LENSIM_EINVAL, "workspace must be 256-byte aligned");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  ConvArgs c{};
  c.nx = nx;
  c.ny = ny;
  c.data = data->d_data;
  c.noise = data->d_noise_map;
  c.expo = data->d_exposure_map;
  c.mask = data->d_mask;
  c.exposure_time = data->exposure_time;
  c.bkg2 = data->background_rms * data->background_rms;
  c.inv_t = 1.0 / data->exposure_time;
  c.dstride = data->image_stride;
  double *partial = static_cast<double *>(ws);
  const int nblk = (nx * ny + 255) / 256;
  CallRanges cr;
  const size_t npix = size_t(nx) * ny;
  const size_t nd = data->image_stride ? size_t(n_img - 1) * size_t(data->image_stride) + npix : npix;
  cr.add(data->d_data, nd * sizeof(double));
  cr.add(data->d_noise_map, nd * sizeof(double));
  cr.add(data->d_exposure_map, npix * sizeof(double));
  cr.add(data->d_mask, npix * sizeof(double));
  cr.add(d_model, size_t(n_img) * npix * (precision == LENSIM_FP64 ? sizeof(double) : sizeof(float)));
  cr.add(d_logl, size_t(n_img) * sizeof(double));
  cr.add(ws, need);
  int rc = cr.begin(st);
  if (rc) return rc;
  if (precision == LENSIM_FP64)
    data_chi2_kernel<double><<<dim3(nblk, n_img), 256, 0, st>>>(c, static_cast<const double *>(d_model), partial);
  else
    data_chi2_kernel<float><<<dim3(nblk, n_img), 256, 0, st>>>(c, static_cast<const float *>(d_model), partial);
  if ((rc = check_launch("data_chi2_kernel"))) return cr.end(st, rc);
  logl_kernel<<<n_img, 64, 0, st>>>(partial, nblk, nullptr, d_logl);
  return cr.end(st, check_launch("logl_kernel"));
}

size_t lensim_linear_workspace_size(const lensim_model *model, const lensim_grid *grid, const lensim_psf *psf,
                                    int32_t n_img, int32_t precision) {
  ModelArgs m;
  if (model_args(model, m) || !grid) return 0;
  GridArgs g;
  SSPlan ss;
  int kx = 1, ky = 1, edge = 0;
  if (grid_args(grid, g) || psf_ss(psf, g, 0, ss) || psf_dims(psf, 0, kx, ky, edge)) return 0;
  return lin_layout(m, g.nx, g.ny, kx, ky, n_img, precision, ss, m.n_source + m.n_light).total;
}

int lensim_linear_solve(const lensim_model *model, const lensim_grid *grid, const lensim_psf *psf,
                        const lensim_data *data, const double *d_params, int32_t n_img, int32_t precision,
                        int32_t source_marg, double linear_prior, double *d_amp, double *d_logl, void *d_model_out,
                        double *d_cov, void *d_response_out, void *ws, size_t ws_bytes, void *stream) {
  ModelArgs m;
  int rc = model_args(model, m);
  if (rc) return rc;
  GridArgs g;
  if ((rc = grid_args(grid, g))) return rc;
  int kx, ky, edge;
  if ((rc = psf_dims(psf, 0, kx, ky, edge))) return rc;
  SSPlan ss;
  if ((rc = psf_ss(psf, g, 0, ss))) return rc;
  const int n_lin = m.n_source + m.n_light;
  if (n_lin == 0) return fail(LENSIM_EINVAL, "the linear solve needs at least one light profile");
  if (n_lin > kMaxLin) return fail(LENSIM_EUNSUPPORTED, "at most %d linear amplitudes (got %d)", kMaxLin, n_lin);
  if (!data || !data->d_data) return fail(LENSIM_EINVAL, "data image is NULL");
  if (!data->d_noise_map && !data->d_exposure_map && !(data->exposure_time > 0.0))
    return fail(LENSIM_EINVAL, "need a noise map, an exposure map or a positive exposure time");
  if (data->image_stride != 0 && data->image_stride < int64_t(g.nx) * g.ny)
    return fail(LENSIM_EINVAL, "image_stride %lld is smaller than an image", (long long)data->image_stride);
  if (n_img < 0) return fail(LENSIM_EINVAL, "negative n_img");
  if (n_img == 0) return LENSIM_OK;
  if (n_img > 65535) return fail(LENSIM_EINVAL, "n_img %d exceeds 65535 per call", n_img);
  if (!d_logl || !d_params) return fail(LENSIM_EINVAL, "NULL buffer");
  if (precision != LENSIM_FP64 && precision != LENSIM_MIXED) return fail(LENSIM_EINVAL, "bad precision");
  const LinLayout LL = lin_layout(m, g.nx, g.ny, kx, ky, n_img, precision, ss, n_lin);
  if (LL.total > ws_bytes)
    return fail(LENSIM_EWORKSPACE, "workspace of %zu B is smaller than the %zu B needed", ws_bytes, LL.total);
  if (!ws || (reinterpret_cast<uintptr_t>(ws) & 255)) return fail(LENSIM_EINVAL, "workspace must be 256-byte aligned");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  unsigned char *w = static_cast<unsigned char *>(ws);
  const size_t tsz = precision == LENSIM_FP64 ? sizeof(double) : sizeof(float);
  const size_t npix = size_t(g.nx) * g.ny;
  CallRanges cr;
  add_inputs(cr, model, m, d_params, n_img, grid, psf, data, g.nx, g.ny);
  cr.add(d_amp, size_t(n_img) * n_lin * sizeof(double));
  cr.add(d_logl, size_t(n_img) * sizeof(double));
  cr.add(d_model_out, size_t(n_img) * npix * tsz);
  cr.add(d_cov, size_t(n_img) * n_lin * n_lin * sizeof(double));
  cr.add(d_response_out, size_t(n_lin) * n_img * npix * tsz);
  cr.add(ws, LL.total);
  if ((rc = cr.begin(st))) return rc;
  if (precision == LENSIM_FP64)
    rc = run_linear<double>(m, g, psf, kx, ky, edge, ss, data, d_params, n_img, source_marg, linear_prior, d_amp,
                            d_logl, static_cast<double *>(d_model_out), d_cov,
                            static_cast<double *>(d_response_out), w, LL, st);
  else
    rc = run_linear<float>(m, g, psf, kx, ky, edge, ss, data, d_params, n_img, source_marg, linear_prior, d_amp,
                           d_logl, static_cast<float *>(d_model_out), d_cov, static_cast<float *>(d_response_out), w,
                           LL, st);
  return cr.end(st, rc);
}

size_t lensim_grad_workspace_size(const lensim_model *model, const lensim_grid *grid, const lensim_psf *psf,
                                  int32_t n_img, int32_t precision) {
  ModelArgs m;
  if (model_args(model, m) || !grid) return 0;
  int kx = 1, ky = 1, edge = 0;
  if (psf_dims(psf, 0, kx, ky, edge)) return 0;
  GridArgs g;
  SSPlan ss;
  if (grid_args(grid, g) || psf_ss(psf, g, 0, ss)) return 0;
  return grad_layout(m, grid->nx, grid->ny, kx, ky, n_img, precision, edge, ss, g.s).total;
}

int lensim_loglike_grad(const lensim_model *model, const lensim_grid *grid, const lensim_psf *psf,
                        const lensim_data *data, const double *d_params, int32_t n_img, int32_t precision,
                        double *d_logl, double *d_grad, void *ws, size_t ws_bytes, void *stream) {
  ModelArgs m;
  int rc = model_args(model, m);
  if (rc) return rc;
  GridArgs g;
  if ((rc = grid_args(grid, g))) return rc;
  int kx, ky, edge;
  if ((rc = psf_dims(psf, 0, kx, ky, edge))) return rc;
  SSPlan ss;
  if ((rc = psf_ss(psf, g, 0, ss))) return rc;
  if (!data || !data->d_data) return fail(LENSIM_EINVAL, "data image is NULL");
  if (!data->d_noise_map && !data->d_exposure_map && !(data->exposure_time > 0.0))
    return fail(LENSIM_EINVAL, "need a noise map, an exposure map or a positive exposure time");
  if (data->image_stride != 0 && data->image_stride < int64_t(g.nx) * g.ny)
    return fail(LENSIM_EINVAL, "image_stride %lld is smaller than an image", (long long)data->image_stride);
  if (n_img < 0) return fail(LENSIM_EINVAL, "negative n_img");
  if (n_img == 0) return LENSIM_OK;
  if (n_img > 65535 || m.n_prof > 65535) return fail(LENSIM_EINVAL, "batch too large");
  if (m.mp_n && int64_t(g.nx) * g.ny * g.s * g.s >= (int64_t(1) << 30))
    return fail(LENSIM_EINVAL, "multi-plane gradients take fewer than 2^30 rays per image");
  if (!d_logl || !d_grad || !d_params) return fail(LENSIM_EINVAL, "NULL buffer");
  if (precision != LENSIM_FP64 && precision != LENSIM_MIXED) return fail(LENSIM_EINVAL, "bad precision");
  const Layout L = grad_layout(m, g.nx, g.ny, kx, ky, n_img, precision, edge, ss, g.s);
  if ((rc = check_ws(L, ws, ws_bytes))) return rc;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  unsigned char *w = static_cast<unsigned char *>(ws);
  CallRanges cr;
  add_inputs(cr, model, m, d_params, n_img, grid, psf, data, g.nx, g.ny);
  cr.add(d_logl, size_t(n_img) * sizeof(double));
  cr.add(d_grad, size_t(n_img) * m.n_prof * LENSIM_NPARAM * sizeof(double));
  cr.add(ws, L.total);
  if ((rc = cr.begin(st))) return rc;
  if (precision == LENSIM_FP64)
    rc = run_grad<double>(m, g, psf, kx, ky, edge, ss, data, d_params, n_img, d_logl, d_grad, w, L, st);
  else
    rc = run_grad<float>(m, g, psf, kx, ky, edge, ss, data, d_params, n_img, d_logl, d_grad, w, L, st);
  return cr.end(st, rc);
}

size_t lensim_noalloc_scratch_bytes(void) { return kScratchBytes; }

int lensim_loglike_noalloc(const lensim_model *model, const lensim_grid *grid, const lensim_psf *psf,
                           const lensim_data *data, const double *d_params, int32_t n_img, int32_t precision,
                           double *d_logl, void *d_model_out, void *stream) {
  if (n_img > 0) {
    const size_t need = lensim_workspace_size(model, grid, psf, n_img, precision);
    if (need == 0)  // a bad argument: lensim_loglike's own checks name it, before any device work
      return lensim_loglike(model, grid, psf, data, d_params, n_img, precision, d_logl, d_model_out, nullptr, 0,
                            stream);
    if (need > kScratchBytes)
      return fail(LENSIM_EWORKSPACE,
                  "the call needs %zu B of scratch memory; lensim_loglike_noalloc holds %zu B (split the batch, "
                  "or call lensim_loglike with a workspace)",
                  need, kScratchBytes);
  }
  void *ws = nullptr;
  const int rc = scratch_on_device(&ws);
  if (rc) return rc;
  return lensim_loglike(model, grid, psf, data, d_params, n_img, precision, d_logl, d_model_out, ws, kScratchBytes,
                        stream);
}

// ------------------------------------------------------ graph capture ---
struct lensim_graph_s {
  hipGraph_t graph;
  hipGraphExec_t exec;
};

int lensim_graph_capture_loglike(const lensim_model *model, const lensim_grid *grid, const lensim_psf *psf,
                                 const lensim_data *data, const double *d_params, int32_t n_img, int32_t precision,
                                 double *d_logl, void *d_model_out, void *ws, size_t ws_bytes, void *stream,
                                 lensim_graph *out) {
  if (!out) return fail(LENSIM_EINVAL, "graph handle pointer is NULL");
  *out = nullptr;
  if (!stream) return fail(LENSIM_EINVAL, "graph capture needs a stream other than the NULL stream");
  if (n_img <= 0) return fail(LENSIM_EINVAL, "graph capture needs n_img > 0");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  hipError_t e = hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal);
  if (e != hipSuccess) return hip_fail(e, "hipStreamBeginCapture");
  g_capturing = true;
  const int rc = lensim_loglike(model, grid, psf, data, d_params, n_img, precision, d_logl, d_model_out, ws,
                                ws_bytes, stream);
  g_capturing = false;
  hipGraph_t graph = nullptr;
  e = hipStreamEndCapture(st, &graph);  // ends the capture whatever the call returned
  if (rc != LENSIM_OK) {
    if (graph) (void)hipGraphDestroy(graph);
    return rc;
  }
  if (e != hipSuccess) return hip_fail(e, "hipStreamEndCapture");
  hipGraphExec_t exec = nullptr;
  e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  if (e != hipSuccess) {
    (void)hipGraphDestroy(graph);
    return hip_fail(e, "hipGraphInstantiate");
  }
  lensim_graph g = static_cast<lensim_graph>(malloc(sizeof(lensim_graph_s)));
  if (!g) {
    (void)hipGraphExecDestroy(exec);
    (void)hipGraphDestroy(graph);
    return fail(LENSIM_EINVAL, "out of host memory");
  }
  g->graph = graph;
  g->exec = exec;
  *out = g;
  return LENSIM_OK;
}

int lensim_graph_launch(lensim_graph g, void *stream) {
  if (!g) return fail(LENSIM_EINVAL, "graph is NULL");
  const hipError_t e = hipGraphLaunch(g->exec, reinterpret_cast<hipStream_t>(stream));
  if (e != hipSuccess) return hip_fail(e, "hipGraphLaunch");
  return LENSIM_OK;
}

int lensim_graph_destroy(lensim_graph g) {
  if (!g) return LENSIM_OK;
  const hipError_t e1 = hipGraphExecDestroy(g->exec);
  const hipError_t e2 = hipGraphDestroy(g->graph);
  free(g);
  if (e1 != hipSuccess) return hip_fail(e1, "hipGraphExecDestroy");
  if (e2 != hipSuccess) return hip_fail(e2, "hipGraphDestroy");
  return LENSIM_OK;
}

}  // extern "C"
