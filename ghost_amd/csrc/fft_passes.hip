// fft_passes.hip -- FFT pass kernels for GHOST's fftp layouts on gfx950.
//
// Every pass streams whole lines through registers (LineFFT) and uses LDS only
// for the Stockham exchanges and for the tile transposes that connect the
// x-contiguous real layout, the ky-contiguous intermediate Q and the
// kz-contiguous spectral layout S.  The transposes are fused into the first
// (load) or last (store) step of the x and z passes; global accesses are
// either whole contiguous lines or L-point chunks along ky (L*16 bytes).
#include <type_traits>

#include "fft_engine.h"
#include "fft_passes.h"

// The launchers are split into parts (GHX_PART=1..9) so the build compiles
// them in parallel; each part instantiates only the kernels it launches.
#ifndef GHX_PART
#error "compile with -DGHX_PART=1..9"
#endif

namespace ghx {

// Sizes with a compiled schedule (complex line lengths).
#define GHX_SIZES(X) \
  X(2) X(3) X(4) X(5) X(6) X(8) X(10) X(12) X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384) X(512) X(1024)

#if GHX_PART == 1
bool fft_size_supported(int n) {
  switch (n) {
#define GHX_CASE(n_) case n_:
    GHX_SIZES(GHX_CASE)
#undef GHX_CASE
    return true;
  default:
    return false;
  }
}

#endif

static size_t g_max_lds = 0;
static size_t max_lds() {
  if (!g_max_lds) {
    int dev = 0, v = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || v <= 0)
      v = 65536;
    g_max_lds = (size_t)v;
  }
  return g_max_lds;
}

// ---------------------------------------------------------------------------
// Launch shapes.  The z and y passes run tiles of L lines x T lanes
// (__launch_bounds__(kTileBound)); the x passes run blocks of whole rows
// (__launch_bounds__(kRowBound)).  Both shapes are computed here, for the
// launchers and for ghx_pass_shape, and every launch is checked against them
// before it is issued (launch_check).
// ---------------------------------------------------------------------------
constexpr unsigned kTileBound = 512;
constexpr unsigned kRowBound = 256;
constexpr int kMaxTile = 32;  // the tile passes keep one bit per line in a 32-bit mask

struct PassShape {
  int lines;       // tile width L, or rows per block
  unsigned block;  // lanes per block
  size_t lds;      // dynamic LDS bytes
};

// Tile width: a power of two no wider than `want`, kMaxTile and the lines
// there are, with L * T <= kTileBound and L rows of `rowslots` points in LDS.
static int pick_L(int T, int rowslots, int nlines, int want, size_t ldsmax) {
  int L = 1;
  while (L * 2 <= want && L * 2 <= kMaxTile) L *= 2;
  while (L > 1 && ((size_t)L * rowslots * sizeof(cplx) > ldsmax || L * T > (int)kTileBound)) L >>= 1;
  if (L > nlines) {
    L = 1;
    while (L * 2 <= nlines) L *= 2;
  }
  return L < 1 ? 1 : L;
}
static PassShape tile_shape(int T, int rowslots, int nlines, int want, size_t ldsmax) {
  const int L = pick_L(T, rowslots, nlines, want, ldsmax);
  return PassShape{L, (unsigned)(L * T), (size_t)L * rowslots * sizeof(cplx)};
}
// The wide y inverse: 8-line tiles (the kernel stores 128-byte chunks); the
// launcher takes it only where their LDS fits, else the tile pass.
static PassShape wide_shape(int TW, int rowslots, int nlines) {
  (void)nlines;
  return PassShape{8, (unsigned)(8 * TW), (size_t)8 * rowslots * sizeof(cplx)};
}
// Rows per block of an x pass: kRowBound lanes, fewer rows when their LDS
// lines would not fit (the kernels read the row count from blockDim.x / T).
// Rows synchronise by wavefront, so launches of up to 9 wavefronts per CU go
// out one wavefront per block, which spreads them over all CUs (blocks of 32 rows
// of 64 points otherwise leave half of them idle at 64^3).  Measured,
// blocks of 256 -> 64 lanes, us: X cross 11.2 -> 8.4 at 32^3, 11.4 -> 10.6 at
// 64^3, 12.6 -> 11.8 at 128 x 64 x 32, 23.1 -> 22.1 at 384 x 48 x 48, tracers'
// inverse 14.2 -> 12.0 at 96^3 (2304 wavefronts); the same at 128^3 (4096).
static PassShape row_shape(int T, int rowslots, size_t ldsmax, long rows = 1L << 30) {
  const int lanes = rows * T <= 64 * 2304L ? 64 : (int)kRowBound;
  int r = lanes / T;
  if (r < 1) r = 1;
  while (r > 1 && (size_t)r * rowslots * sizeof(cplx) > ldsmax) r >>= 1;
  return PassShape{r, (unsigned)(r * T), (size_t)r * rowslots * sizeof(cplx)};
}

constexpr int zrk_groups(int KIND) { return KIND == 2 ? 4 : 3; }
constexpr unsigned zrk_bound(int KIND) { return KIND == 2 ? 512 : 768; }
// Launch of k_zrk (KIND 0 HD, 1 MHD, 2 Boussinesq; one group of lanes per
// component): tiles of up to `want` lines, as many as G groups of T lanes per
// line leave within the kernel's bound and the LDS of one block.
static PassShape zrk_shape(int G, int T, unsigned bound, int rowslots, int nlines, int want, size_t ldsmax) {
  int L = 1;
  while (L * 2 <= want && L * 2 <= kMaxTile && L * 2 <= nlines && (unsigned)(G * L * 2 * T) <= bound &&
         (size_t)G * L * 2 * rowslots * sizeof(cplx) <= ldsmax)
    L *= 2;
  return PassShape{L, (unsigned)(G * L * T), (size_t)G * L * rowslots * sizeof(cplx)};
}
// The schedules of the grouped updates are those of the large launches' updates,
// so that a run's rounding does not hang on its size: four points per lane for
// MHD where a length has that schedule and for HD's 512-point lines (and others
// on request, FFTCtx::sched), 64 and 512 points 1.84 and 2.52e-16 of rounding a
// line against 2.52 and 3.42 on the default schedule.
template <int N> constexpr bool has_low() { return FFTCfgLow<N>::E != FFTCfg<N>::E; }
template <int N, int KIND>
using ZrkCfg = typename std::conditional<has_low<N>() && (KIND == 1 || (KIND == 0 && N == 512)), FFTCfgLow<N>, FFTCfgMix<N>>::type;

// The small planes' kernel (k_xyplane): kRowBound lanes, a padded x line for
// every T of them and the plane's nx / 2 + 1 y lines.
#define GHX_PLANE_SIZES(X) X(24) X(32) X(48) X(64)
static bool plane_size(int n) {
  switch (n) {
#define GHX_CASE(n_) case n_:
    GHX_PLANE_SIZES(GHX_CASE)
#undef GHX_CASE
    return true;
  default:
    return false;
  }
}
static constexpr PassShape plane_shape(int nx, int ny) {
  const int Tx = nx % 3 == 0 ? nx / 6 : nx / 8;
  const int rows = (int)kRowBound / Tx;
  return PassShape{rows, kRowBound, ((size_t)rows * lds_line_stride(nx) + (size_t)(nx / 2 + 1) * lds_line_stride(ny)) * sizeof(cplx)};
}

// Whether a device gives the LDS of these launches; where it does not, the
// separate x and y passes and the updates that take one component after another run.
// (gfx950's 160 KiB hold them all; 64 KiB refuse planes of 64 x 48 and 64 x 64
// points and the Boussinesq update of 1024-point lines.)
static bool takes_plane(int nx, int ny, size_t ldsmax) { return plane_shape(nx, ny).lds <= ldsmax; }
static bool takes_zrk(int G, int rowslots, size_t ldsmax) { return (size_t)G * rowslots * sizeof(cplx) <= ldsmax; }

// Modes 0 and 3 hold one field: 12 points per lane for the long 3 * 2^k lines
// (the spline pass 27 us against 30 on the mixed stages at 192^3, 153 against
// 217 at 384^3); the mixed stages below.
template <int N>
using ZInvCfg = typename std::conditional<FFTCfgMid<N>::E != FFTCfg<N>::E && (N >= 192), FFTCfgMid<N>, FFTCfgMix<N>>::type;
// Schedules of the 3 * 2^k lines.  The y inverse is bound by its stores from 96
// points on and takes 12 points per lane (six fields: mixed stages 100 against
// 70 us at 192^3, 17.6 against 13.4 at 96^3); so does the y forward from 192 on
// (45 against 43 us at 192^3), and keeps 6 at 96 (mixed 13.7 against 12.6 for
// four fields, 12 points 13 against 12).  Shorter lines take the mixed stages
// (9.0 -> 8.3 us at 48^3).
template <int N>
using YInvCfg = typename std::conditional<FFTCfgMid<N>::E != FFTCfg<N>::E, FFTCfgMid<N>, FFTCfgMix<N>>::type;
template <int N> struct YFwd { using Cfg = YInvCfg<N>; };
template <> struct YFwd<96> { using Cfg = FFTCfg<96>; };
template <int N> using YFwdCfg = typename YFwd<N>::Cfg;
// The Boussinesq update on 192-point lines spills on the mixed stages (70 -> 84
// us at 192^3) and keeps 6 points per lane; 384 and 96 points gain (64 -> 50 us
// at 96 x 96 x 384, 15 -> 14 at 96^3).
template <int N>
using ZBoussCfg = typename std::conditional<N == 192, FFTCfg<N>, FFTCfgMix<N>>::type;
// Launches of up to this many kept lines (13 per CU; 96^3 has 3168, 128^3
// 5504) leave the GPU waiting on the chain inside a block, so a block is given
// one field or one component instead of all of them in turn.  Measured at
// 32^3, 64^3, 96^3 and 128^3 (us, with ~3 of event overhead): six-field y
// inverse 12.9 -> 7.3, 14.4 -> 9.7, 20.6 -> 13.3, 23.8 -> 27.7; curl z inverse
// 11.8 -> 9.4, 12.9 -> 11.7, 17.8 -> 17.4, 20.9 -> 30.1; HD update 14.2 -> 8.8,
// 15.9 -> 10.8, 16.6 -> 13.2, 23.3 -> 24.7.
// Long z lines turn earlier: what one field per block reads and transforms
// again grows with the line.  All fields in turn | one per block, curl and
// update: 256 points, 704 lines 17.5 | 15.0 and 20.4 | 15.0, 1408 lines 18.7 |
// 22.1 and 22.2 | 24.0; 384 points, 704 lines 18.5 | 17.8, 1408 23.7 | 26.5; 512
// points, 352 lines 17.9 | 15.8, 704 18.9 | 22.4, 3168 28.2 | 50.2; 1024 points,
// 352 lines 33.0 | 30.2, 704 35.0 | 46.7.  (192 points: 18.3 | 17.4 at 1408 lines,
// 23.1 | 21.5 at 3168, but 23.5 | 25.7 at 2752; whole steps of HD, MHD and
// Boussinesq gain or lose up to 7% either way and keep the limit.)  So beyond
// 192 points the limit is a volume, and never below 384 lines, which leave CUs
// without a tile.  Fields that are only transformed, and a curl alone, read
// little twice and keep kSmallLines at any length (c2r of 64 x 32 x 512 16.4 |
// 15.1, diagnostics of 64 x 64 x 1024 444 | 419).
constexpr long kSmallLines = 3328;
static constexpr long small_z_lines(int nz) {
  const long v = 1408L * 192 / nz;
  return nz <= 192 ? kSmallLines : v > 384 ? v : 384;
}
// The y passes read nothing twice; the lines of 384 points (six fields in turn |
// one per block 38.3 | 25.5 at 1408 lines, 45.0 | 52.9 at 3168) and of 1024
// (30.9 | 26.6 at 352, 33.5 | 40.3 at 704) turn earlier all the same, 512 and
// less not below 3328 (52.3 | 54.9 at 3168 of 512).
static constexpr long small_y_lines(int ny) { return ny > 512 ? 512 : ny == 384 ? 2112 : kSmallLines; }

// Long y inverses are split by field too, all tiles of one field before the
// next's, where that was measured to gain.  All fields in turn | split, us: up to
// 96 points 41.1 | 39.1 (6 fields of 256 x 64 x 256), 49.9 | 43.4 (256 x 96 x 192);
// 192 points 113.9 | 110.7 (9 fields of 192^3), 71.1 | 71.2 (6), 40.4 | 40.6 (3); six
// and more fields of 256 and 384 points on long launches 179.8 | 171.6 (256^3),
// 650 | 611 (384^3), but 77.8 | 80.5 (256 x 256 x 128), 215.9 | 249.4 (512 x 384 x
// 96), and three 74.5 | 83.5 (256^3), 145.8 | 166.2 (384 x 384 x 192); not 128
// points (78.7 | 82.1 for 256 x 128 x 256), 512 (2%) or 1024 (the same).  45 | 46
// us at 128 x 256 x 128 (5504 lines), 39 | 40 at 192 x 128 x 128 (8320).  Without
// pruning three fields gain too: 172 | 166 (256^3), 286 | 269 (384 x 384 x 192), 71 |
// 68 (256 x 256 x 128).
static constexpr bool long_y(int ny, int nf, long lines, bool pruned) {
  if (!pruned) return lines >= 10000 && ny != 512;
  if (ny <= 96 || ny == 192) return lines >= 10000;
  return (ny == 256 || ny == 384) && nf >= 6 && lines >= 20000;
}

// Refuses, before it is issued, a launch that its kernel was not built for:
// more lanes than its __launch_bounds__ or than the code object's maximum
// work-group size, a block that is not whole lines of T lanes, a tile wider
// than the line masks, or more LDS than the device gives one block.
static hipError_t launch_check(unsigned most, const char *name, const PassShape &s, unsigned bound, int T, bool tile) {
  const char *why = nullptr;
  if (s.block < 1 || s.block > bound) why = "more lanes than the kernel's launch bounds";
  else if (T < 1 || s.block % (unsigned)T) why = "a block that is not whole lines";
  else if (tile && (s.lines < 1 || s.lines > kMaxTile || (s.lines & (s.lines - 1)))) why = "a tile width that is not a power of two up to 32";
  else if (s.lds > max_lds()) why = "more LDS than one block may hold";
  else if (most && s.block > most) why = "more lanes than the code object allows";
  if (!why) return hipSuccess;
  fprintf(stderr, "ghx: refused launch of %s: %s (block %u, %d lines, T %d, LDS %zu bytes, bound %u)\n", name, why,
          s.block, s.lines, T, s.lds, bound);
  return hipErrorInvalidConfiguration;
}
// A kernel's maximum work-group size (0: unknown), asked for once per kernel: it
// is a constant of the code object, and asking at each launch is host time that
// the smallest transforms wait for (r2c of 32^3: 12.2 -> 9.8 us of host time a call).
static unsigned kernel_most(const void *kern) {
  hipFuncAttributes a;
  return hipFuncGetAttributes(&a, kern) == hipSuccess && a.maxThreadsPerBlock > 0 ? (unsigned)a.maxThreadsPerBlock : 0;
}
#define GHX_LAUNCH_CHECK(kern, s, bound, T, tile)                                              \
  do {                                                                                         \
    static const unsigned most_ = kernel_most((const void *)(kern));                           \
    const hipError_t ce_ = launch_check(most_, #kern, (s), (bound), (T), (tile));              \
    if (ce_ != hipSuccess) return ce_;                                                         \
  } while (0)

#define GHX_X2_SIZES(X) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384) X(512)
static bool x2_size(int nx) {
  switch (nx) {
#define GHX_CASE(n_) case n_:
    GHX_X2_SIZES(GHX_CASE)
#undef GHX_CASE
    return true;
  default:
    return false;
  }
}

#if GHX_PART == 1
// The launch shape a pass of line length n takes for `nlines` lines along the
// tiled axis, a requested tile width `want` (as the GHX_LZ/GHX_LY knobs and the
// autotuner give it) and a device LDS limit; then the check the launchers
// apply.  Host-only.  Kinds: 0 z and y tile passes on the default schedule; 1
// the Boussinesq z forward, whose LDS rows hold n more points; 2 the wide y
// inverse; 3 two-for-one x passes (n = nx) and 4 half-length x passes (n =
// nx/2) in full blocks; 5, 6, 7 the grouped HD, MHD and Boussinesq updates; 8
// the small planes' kernel (n = nx, nlines = ny); 10 and 11 the x passes of 3
// and 4 for nlines rows; 12 the y inverse, 13 the y forward and 14 the z
// inverse of separate fields on their own schedules; 15 and 16: *lines is the
// number of kept lines up to which a z or y launch takes one field per block; 17
// and 18: *lines is 1 where a pruned or whole y inverse of want fields and nlines
// kept lines beyond that takes one too (nothing else is set).  Kinds 5 to 8 give -3 where
// the launcher takes the other kernels.
extern "C" int ghx_pass_shape(int kind, int n, int nlines, int want, long long ldsmax, int *lines, int *block,
                              long long *lds, int *lanes) {
  int T = 0, rows = 0;
  switch (n) {
#define GHX_CASE(n_)                                                                   \
  case n_:                                                                             \
    rows = lds_line_stride(n_);                                                        \
    if (kind == 0) T = FFTCfg<n_>::T;                                                  \
    if (kind == 1) T = FFTCfg<n_>::T, rows += n_;                                      \
    if (kind == 2 && FFTCfgWide<n_>::E != FFTCfg<n_>::E) T = FFTCfgWide<n_>::T;        \
    if ((kind == 3 || kind == 10) && x2_size(n_)) T = FFTCfg<n_>::T;                   \
    if (kind == 4 || kind == 11) T = FFTCfgLow<n_>::T;                                 \
    if (kind == 5) T = ZrkCfg<n_, 0>::T;                                               \
    if (kind == 6) T = ZrkCfg<n_, 1>::T;                                               \
    if (kind == 7) T = ZrkCfg<n_, 2>::T;                                               \
    if (kind == 8 && plane_size(n_) && plane_size(nlines)) T = FFTCfgMix<n_>::T;       \
    if (kind == 12) T = YInvCfg<n_>::T;                                                \
    if (kind == 13) T = YFwdCfg<n_>::T;                                                \
    if (kind == 14) T = ZInvCfg<n_>::T;                                                \
    break;
    GHX_SIZES(GHX_CASE)
#undef GHX_CASE
  default:
    break;
  }
  if ((kind == 15 || kind == 16) && rows > 0 && lines) {
    *lines = (int)(kind == 15 ? small_z_lines(n) : small_y_lines(n));
    return 0;
  }
  if ((kind == 17 || kind == 18) && rows > 0 && lines) {
    *lines = long_y(n, want, nlines, kind == 17) ? 1 : 0;
    return 0;
  }
  if (T <= 0 || nlines < 1 || ldsmax <= 0) return -1;
  PassShape s;
  unsigned bound = kTileBound;
  switch (kind) {
  case 2: s = wide_shape(T, rows, nlines); break;
  case 3: case 4: s = row_shape(T, rows, (size_t)ldsmax), bound = kRowBound; break;
  case 5: case 6: case 7:
    if (!takes_zrk(zrk_groups(kind - 5), rows, (size_t)ldsmax)) return -3;
    bound = zrk_bound(kind - 5);
    s = zrk_shape(zrk_groups(kind - 5), T, bound, rows, nlines, want, (size_t)ldsmax);
    break;
  case 8:
    if (!takes_plane(n, nlines, (size_t)ldsmax)) return -3;
    s = plane_shape(n, nlines), bound = kRowBound; break;
  case 10: case 11: s = row_shape(T, rows, (size_t)ldsmax, nlines), bound = kRowBound; break;
  default: s = tile_shape(T, rows, nlines, want, (size_t)ldsmax); break;
  }
  if (lines) *lines = s.lines;
  if (block) *block = (int)s.block;
  if (lds) *lds = (long long)s.lds;
  if (lanes) *lanes = T;
  const bool tile = kind <= 2 || (kind >= 5 && kind <= 7) || kind >= 12;
  if (s.block < 1 || s.block > bound || s.block % (unsigned)T || s.lds > (size_t)ldsmax) return -2;
  if (tile && (s.lines < 1 || s.lines > kMaxTile || (s.lines & (s.lines - 1)))) return -2;
  return 0;
}
#endif

// Tile widths (lines per block along ky) for the z and x passes; overridable
// with GHX_LZ / GHX_LX for tuning sweeps.
static int tile_want(const char *env, int dflt) {
  const char *e = getenv(env);
  int v = e ? atoi(e) : 0;
  return v > 0 ? v : dflt;
}

// An on/off switch for measurements: its value when set (0 included), else dflt.
static int env_switch(const char *env, int dflt) {
  const char *e = getenv(env);
  return e && *e ? atoi(e) : dflt;
}

// tile width: the environment override (tuning sweeps), else the context's
// choice, else the built-in default
static int tile_pick(const char *env, int ctx, int dflt) {
  const int e = tile_want(env, 0);
  return e > 0 ? e : (ctx > 0 ? ctx : dflt);
}

// Row lengths with a two-for-one x kernel (a full-length schedule of 6 or 8
// points per lane and at most 64 lanes; ghx_pass_shape takes the same list);
// GHX_XC2=0 selects the half-length kernels instead, for comparisons.
static bool use_x2(int nx) {
  if (env_switch("GHX_XC2", 1) != 1) return false;
  return x2_size(nx);
}

// Built-in tile width: `lines`, or as many more as fill a wavefront (a line of
// few lanes would leave half or more of it idle: 4 lines of 8 lanes).
static constexpr int tile_default(int T, int lines) { return lines * T >= 64 ? lines : 64 / T; }

// What a launch passes for its input's pruning (prune_input): the flag and the
// device word that may clear it.
static int prune_in(const FFTCtx &c, int prune) { return prune == 2 ? (c.dirty ? 1 : 0) : prune; }
static const unsigned *prune_word(const FFTCtx &c, int prune) { return prune == 2 ? c.dirty : nullptr; }
// kx below which a pass reads its input (unless the word says more) and writes its output
static int kx_in(const FFTCtx &c, int prune) { return prune_in(c, prune) ? c.gk.kxact : c.gk.nxh; }
static int kx_out(const FFTCtx &c, int prune) { return prune ? c.gk.kxact : c.gk.nxh; }

static long z_lines(const FFTCtx &c) { return (long)c.gk.kxact * c.gk.ny * c.batch; }
static bool small_z(const FFTCtx &c) { return z_lines(c) <= small_z_lines(c.gk.nz); }
static bool small_y(const FFTCtx &c) { return (long)c.gk.kxact * c.gk.nz * c.batch <= small_y_lines(c.gk.ny); }

template <typename K> static void allow_lds(K kern, size_t bytes) {
  if (bytes > 49152) (void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

// ---------------------------------------------------------------------------
// XCD-aware tile order.  Workgroups are dealt round-robin to the 8 XCDs by
// linear id and each XCD has its own L2.  A tile narrower than a 128-byte
// line shares its lines with the neighbouring tile along the chunked axis, so
// within each group of 16 linear ids the two ids that land on the same XCD
// (b and b+8) are given neighbouring tiles.  Tiles stay spread over the XCDs
// in their natural order, which keeps pruned passes load-balanced, but for rows
// of 16, 32, .. tiles (128, 256, .. ky): there a tile would meet the same XCD in
// every row, and the tiles that pruning empties (the middle third of ky) are
// the same in every row, so two XCDs would idle while two have half as much
// again.  So in the pruned z passes each such row starts one XCD further than
// the last (spread).  us without | with: curl z inverse 119.9 | 81.6 at 256^3, 33.6
// | 24.5 at 128 x 256 x 128, 355 | 293 at 512 x 512 x 256; MHD update 291 | 202 at
// 256^3.  (Without pruning, and in the y passes, whose rows are of other lengths
// and pass all XCDs by themselves, it only costs: one field's z inverse of 64 x
// 64 x 512 14.8 | 17.2, y inverses up to a third.)
// ---------------------------------------------------------------------------
// Member b of a batched launch: every field pointer moves by b * bstride.
// The view reads the pointers from the kernel arguments on each use and adds
// the offset; a shifted copy of the argument that is indexed by a run-time
// field number would be placed in scratch memory.
struct FieldRef {
  const FieldSet &fs;
  size_t off;
  GHX_DEV cplx *operator[](int f) const { return fs.p[f] + off; }
};
struct FieldView {
  FieldRef p;
};
GHX_DEV FieldView batch_view(const FieldSet &fs, unsigned b) { return FieldView{FieldRef{fs, (size_t)b * fs.bstride}}; }

// tile of linear id b among rows of gx tiles, nb in all
__host__ __device__ inline int xcd_order(int b, int row, int gx, int nb, bool spread) {
  if (b >= (nb & ~15)) return b;
  if (spread && (gx & 15) == 0) b = (b & ~7) | ((b + row) & 7);
  return (b & ~15) | ((b & 7) << 1) | ((b >> 3) & 1);
}
GHX_DEV void xcd_tile(int &bx, int &by, bool spread = false) {
  const int b = xcd_order(blockIdx.y * gridDim.x + blockIdx.x, blockIdx.y, gridDim.x, gridDim.x * gridDim.y, spread);
  bx = b % gridDim.x;
  by = b / gridDim.x;
}
#if GHX_PART == 1
extern "C" int ghx_tile_order(int gx, int rows, int spread, int *tile) {
  if (gx < 1 || rows < 1 || !tile) return -1;
  for (int b = 0; b < gx * rows; ++b) tile[b] = xcd_order(b, b / gx, gx, gx * rows, spread != 0);
  return 0;
}
#endif

// ---------------------------------------------------------------------------
// Tile helpers (block = L lines x T lanes; line lt = threadIdx.x / T)
// ---------------------------------------------------------------------------

// Store the L lines of a block (kept in LDS rows) with the line index
// fastest: point p of line l goes to dst[p * pstride + l] when keep(l) (the
// dealias pruning and the tile's edge; the loader zero-fills the rest without
// touching memory).  The block is exactly L x T lanes with L a power of two
// and E * T points per row, so every lane moves E points: line
// l = idx & (L - 1), point idx >> log2 L.  The loop stays rolled (G points
// per trip): holding all E points at once costs most y and z kernels a wave
// per SIMD or spills; a caller with registers to spare sets G = E through GW
// (the 512-point curl z inverse, 8 points).  NT selects streaming
// stores: the y inverse (128-byte chunks) gains 10-14% with them, the z
// inverse (64-byte chunks at L = 4) loses 5-11%.
//
// The block is L x T lanes with L a power of two, so l is the same on every
// trip: the keep test is made once per lane, and the LDS reads go in groups
// of G (up to 4; GW > 0 sets it) ahead of their stores, so that a group's
// reads are in flight together instead of each store waiting on its own read.
template <int E, bool NT, int GW = 0, typename Keep>
GHX_DEV void tile_store_rows(const cplx *lds, int stride, int L, cplx *dst, size_t pstride, Keep keep) {
  constexpr int G = GW > 0 ? GW : E % 4 == 0 ? 4 : E % 3 == 0 ? 3 : E % 2 == 0 ? 2 : 1;
  static_assert(E % G == 0, "the group width divides the points per lane");
  const int lsh = 31 - __builtin_clz((unsigned)L);
  if constexpr (G == 1) {
    // one point per trip, the keep test in the loop: the fewest live
    // registers, for kernels at the register limit
#pragma unroll 2
    for (int q = 0; q < E; ++q) {
      const int idx = threadIdx.x + q * blockDim.x;
      const int l = idx & (L - 1);
      const cplx x = lds[l * stride + lds_pad(idx >> lsh)];
      if (keep(l)) c_put<NT>(dst + (size_t)(idx >> lsh) * pstride + l, x);
    }
    return;
  }
  const int l = threadIdx.x & (L - 1);
  if (!keep(l)) return;
  const int p0 = threadIdx.x >> lsh, dp = blockDim.x >> lsh;
  const cplx *src = lds + l * stride;
  cplx *d = dst + (size_t)p0 * pstride + l;
  const size_t dstep = (size_t)dp * pstride;
#pragma unroll 1
  for (int q0 = 0; q0 < E; q0 += G) {
    cplx x[G];
#pragma unroll
    for (int u = 0; u < G; ++u) x[u] = src[lds_pad(p0 + (q0 + u) * dp)];
#pragma unroll
    for (int u = 0; u < G; ++u) c_put<NT>(d + (size_t)(q0 + u) * dstep, x[u]);
  }
}
// Block = L lines x T lanes, E = N / T points per thread.  The E loads of a
// thread issue back to back (lines outside the mask or past ny read line j0,
// inside the tile, and are zeroed by a select), then go to LDS.
template <int E>
GHX_DEV void tile_load_q(cplx *lds, int stride, int L, const cplx *src, size_t pstride, size_t base, int j0, int ny,
                         unsigned lmask = ~0u) {
  cplx w[E];
#pragma unroll
  for (int q = 0; q < E; ++q) {
    const int idx = threadIdx.x + q * blockDim.x;
    const int l = idx % L, p = idx / L;
    const bool inside = j0 + l < ny && ((lmask >> l) & 1u);
    const cplx x = src[base + (size_t)p * pstride + j0 + (inside ? l : 0)];
    w[q] = inside ? x : c_make(0.0, 0.0);
  }
#pragma unroll
  for (int q = 0; q < E; ++q) {
    const int idx = threadIdx.x + q * blockDim.x;
    lds[(idx % L) * stride + lds_pad(idx / L)] = w[q];
  }
}

// tile_load_q in two halves, so that a tile's loads can be in flight while
// the previous tile is transformed: the E loads of a thread into registers,
// then the registers into the LDS rows.
template <int E>
GHX_DEV void tile_fetch_q(cplx (&w)[E], int L, const cplx *src, size_t pstride, size_t base, int j0, int ny,
                          unsigned lmask) {
#pragma unroll
  for (int q = 0; q < E; ++q) {
    const int idx = threadIdx.x + q * blockDim.x;
    const int l = idx % L, p = idx / L;
    const bool inside = j0 + l < ny && ((lmask >> l) & 1u);
    const cplx x = src[base + (size_t)p * pstride + j0 + (inside ? l : 0)];
    w[q] = inside ? x : c_make(0.0, 0.0);
  }
}
template <int E>
GHX_DEV void tile_put_q(cplx *lds, int stride, int L, const cplx (&w)[E]) {
#pragma unroll
  for (int q = 0; q < E; ++q) {
    const int idx = threadIdx.x + q * blockDim.x;
    lds[(idx % L) * stride + lds_pad(idx / L)] = w[q];
  }
}

// A (kx, ky) line carries dealiased modes iff kn2(kx, ky, 0) <= kmax.
GHX_DEV bool line_active(const GridK &g, int i, int j) { return kn2_of(g, i, j, 0) <= g.kmax; }
GHX_DEV unsigned tile_lines_active(const GridK &g, int i, int j0, int L) {
  unsigned m = 0;
  for (int l = 0; l < L; ++l)
    if (j0 + l < g.ny && line_active(g, i, j0 + l)) m |= 1u << l;
  return m;
}

// ---------------------------------------------------------------------------
// Z^-1: S -> Q.  Block = (kx index i, ky chunk j0..j0+L-1).
// ---------------------------------------------------------------------------
// The store half of zinv_emit: the transformed line v (samples as Line holds
// them) into the block's LDS rows, then the tile to Q.
template <int N, int E, typename Cfg = FFTCfgMix<N>, int GW = 0>
GHX_DEV void zinv_store(const cplx (&v)[Line<N, Cfg>::SE], cplx *lds, cplx *row, int stride, int L, int t, cplx *dst,
                        const GridK &g, int i, int j0, unsigned lmask) {
  Line<N, Cfg>::put(v, row, t);
  __syncthreads();
  const int ny = g.ny;
  tile_store_rows<E, false, GW>(lds, stride, L, dst + (size_t)i * ny + j0, (size_t)g.nxh * ny,
                     [=](int l) { return j0 + l < ny && ((lmask >> l) & 1u); });
  __syncthreads();
}

template <int N, int E, typename Cfg = FFTCfgMix<N>, int GW = 0>
GHX_DEV void zinv_emit(const Line<N, Cfg> &fft, cplx (&v)[E], cplx (&x)[Line<N, Cfg>::SE], cplx *lds, cplx *row,
                       int stride, int L, int t, cplx *dst, const GridK &g, int i, int j0, unsigned lmask) {
  fft.inv(v, x, row, t);
  zinv_store<N, E, Cfg, GW>(x, lds, row, stride, L, t, dst, g, i, j0, lmask);
}
template <int N, int E, typename Cfg = FFTCfgMix<N>, int GW = 0>
GHX_DEV void zinv_emit(cplx (&v)[E], cplx *lds, cplx *row, int stride, int L, int t, const Line<N, Cfg> &fft,
                       cplx *dst, const GridK &g, int i, int j0, unsigned lmask) {
  cplx x[Line<N, Cfg>::SE];
  zinv_emit<N, E, Cfg, GW>(fft, v, x, lds, row, stride, L, t, dst, g, i, j0, lmask);
}

// A vector field's z inverse and its curl's with five transforms instead of
// six.  kx and ky are constant along a z line, so Z^-1(i ky a) = i ky Z^-1(a);
// only the kz terms of rotor3 (pseudospec3D_hd.f90:124-200) need transforms of
// their own:
//   curl_x = i ky Z^-1(a_z) - Z^-1(i kz a_y)
//   curl_y = Z^-1(i kz a_x) - i kx Z^-1(a_z)
//   curl_z = i kx Z^-1(a_y) - i ky Z^-1(a_x)
// ax, ay, az are the spectral lines (lane t holding points t + T m); the six
// results go to o[0..2] (a) and o[3..5] (curl a).
template <int N, int E, typename Cfg, int GW = 0>
GHX_DEV void zinv_curl5(cplx (&ax)[E], cplx (&ay)[E], cplx (&az)[E], double kx, double ky, cplx *lds, cplx *row,
                        int stride, int L, int t, const Line<N, Cfg> &fft, cplx *const *o, const GridK &g, int i,
                        int j0, unsigned lmask) {
  using F = Line<N, Cfg>;
  constexpr int T = F::T, SE = F::SE;
  cplx zx[SE], zy[SE], zz[SE];  // Z^-1 of the three
  zinv_emit<N, E, Cfg, GW>(fft, az, zz, lds, row, stride, L, t, o[2], g, i, j0, lmask);
  {
    cplx w[E], x[SE];
#pragma unroll
    for (int m = 0; m < E; ++m) w[m] = c_ik(wavenum(t + T * m, g.nz, g.dkz), ay[m]);
    fft.inv(w, x, row, t);
    if (F::live(t)) {
#pragma unroll
      for (int m = 0; m < SE; ++m) x[m] = c_sub(c_ik(ky, zz[m]), x[m]);
    }
    zinv_store<N, E, Cfg, GW>(x, lds, row, stride, L, t, o[3], g, i, j0, lmask);
  }
  {
    cplx w[E], x[SE];
#pragma unroll
    for (int m = 0; m < E; ++m) w[m] = c_ik(wavenum(t + T * m, g.nz, g.dkz), ax[m]);
    fft.inv(w, x, row, t);
    if (F::live(t)) {
#pragma unroll
      for (int m = 0; m < SE; ++m) x[m] = c_sub(x[m], c_ik(kx, zz[m]));
    }
    zinv_store<N, E, Cfg, GW>(x, lds, row, stride, L, t, o[4], g, i, j0, lmask);
  }
  zinv_emit<N, E, Cfg, GW>(fft, ax, zx, lds, row, stride, L, t, o[0], g, i, j0, lmask);
  zinv_emit<N, E, Cfg, GW>(fft, ay, zy, lds, row, stride, L, t, o[1], g, i, j0, lmask);
  if (F::live(t)) {
#pragma unroll
    for (int m = 0; m < SE; ++m) zx[m] = c_sub(c_ik(kx, zy[m]), c_ik(ky, zx[m]));
  }
  zinv_store<N, E, Cfg, GW>(zx, lds, row, stride, L, t, o[5], g, i, j0, lmask);
}

template <int N, int MODE, typename Cfg = FFTCfgMix<N>>
__global__ __launch_bounds__(kTileBound) void k_zinv(FieldSet in_, FieldSet out_, int nf, GridK g, const cplx *__restrict__ twt,
                                             int prune_, const unsigned *dirty, const double *__restrict__ aux) {
  using F = Line<N, Cfg>;
  const int prune = prune_input(prune_, dirty);
  constexpr int T = F::T, E = F::KE;
  // store groups: the MHD and Boussinesq passes (MODE 2, 5) are at the
  // register limit and spill more with grouped reads; they store one point
  // per trip.  The curl pass takes all 8 points of a lane in one group
  // (0.853 -> 0.812 ms at 512^3, same register count)
  constexpr int SG = MODE == 2 || MODE == 5 ? 1 : (MODE == 1 && E == 8) ? 8 : 0;
  extern __shared__ cplx lds[];
  const int L = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  F fft;  // with this lane's stage roots, loaded once
  fft.load_inv(twt, t);
  const FieldView in = batch_view(in_, blockIdx.z);
  const FieldView out = batch_view(out_, blockIdx.z);
  int bx, by;
  xcd_tile(bx, by, prune != 0);
  const int i = by, j0 = bx * L, j = j0 + lt;
  // prune: the input is dealiased, so only lines inside the dealias disc
  // carry data; only their kept modes are read and only they are written.
  const unsigned lmask = prune ? tile_lines_active(g, i, j0, L) : ~0u;
  if (lmask == 0u) return;  // uniform over the block
  const bool ok = j < g.ny && ((lmask >> lt) & 1u);
  const int stride = lds_line_stride(N);
  cplx *row = lds + lt * stride;
  const size_t sline = ((size_t)i * g.ny + (ok ? j : 0)) * N;
  auto need = [&](int k) { return ok && (!prune || kn2_of(g, i, j, k) <= g.kmax); };
  // every lane loads from inside its line (skipped modes read the line's
  // first point, which the line's own loads fetch anyway) and a select zeroes
  // what is not needed, so the loads of a field issue back to back
  auto load = [&](const cplx *p, int k) {
    const bool nd = need(k);
    const cplx x = p[sline + (nd ? k : 0)];
    return nd ? x : c_make(0.0, 0.0);
  };
  if constexpr (MODE == 0 || MODE == 3) {
    // MODE 3: periodic cubic-spline prefilter.  aux = [sx (nx/2+1) | sy (ny) |
    // sz (nz)] and every mode is scaled by sx[kx] sy[ky] sz[kz] on load.
    double sxy = 1.0;
    if constexpr (MODE == 3) sxy = aux[i] * aux[g.nxh + (ok ? j : 0)];
    for (int f = 0; f < nf; ++f) {
      cplx v[E];
#pragma unroll
      for (int m = 0; m < E; ++m) {
        v[m] = load(in.p[f], t + T * m);
        if constexpr (MODE == 3) v[m] = c_scale(v[m], sxy * aux[g.nxh + g.ny + t + T * m]);
      }
      zinv_emit<N, E, Cfg, SG>(v, lds, row, stride, L, t, fft, out.p[f], g, i, j0, lmask);
    }
  } else if constexpr (MODE == 1) {
    // v -> (v, curl v)
    const double kx = wavenum(i, g.nx, g.dkx), ky = wavenum(j, g.ny, g.dky);
    cplx vx[E], vy[E], vz[E];
#pragma unroll
    for (int m = 0; m < E; ++m) {
      vx[m] = load(in.p[0], t + T * m);
      vy[m] = load(in.p[1], t + T * m);
      vz[m] = load(in.p[2], t + T * m);
    }
    cplx *const o[6] = {out.p[0], out.p[1], out.p[2], out.p[3], out.p[4], out.p[5]};
    zinv_curl5<N, E, Cfg, SG>(vx, vy, vz, kx, ky, lds, row, stride, L, t, fft, o, g, i, j0, lmask);
  } else if constexpr (MODE == 2) {
    // (v, A) -> (v, curl v, b = curl A, curl b)
    const double kx = wavenum(i, g.nx, g.dkx), ky = wavenum(j, g.ny, g.dky);
    {
      cplx vx[E], vy[E], vz[E];
#pragma unroll
      for (int m = 0; m < E; ++m) {
        vx[m] = load(in.p[0], t + T * m);
        vy[m] = load(in.p[1], t + T * m);
        vz[m] = load(in.p[2], t + T * m);
      }
      cplx *const o[6] = {out.p[0], out.p[1], out.p[2], out.p[3], out.p[4], out.p[5]};
      zinv_curl5<N, E, Cfg, SG>(vx, vy, vz, kx, ky, lds, row, stride, L, t, fft, o, g, i, j0, lmask);
    }
    // b = curl A per mode (rotor3), then b and curl b
    cplx bx[E], by[E], bz[E];
#pragma unroll
    for (int m = 0; m < E; ++m) {
      const double kz = wavenum(t + T * m, g.nz, g.dkz);
      const cplx ax = load(in.p[3], t + T * m), ay = load(in.p[4], t + T * m), az = load(in.p[5], t + T * m);
      bx[m] = c_sub(c_ik(ky, az), c_ik(kz, ay));
      by[m] = c_sub(c_ik(kz, ax), c_ik(kx, az));
      bz[m] = c_sub(c_ik(kx, ay), c_ik(ky, ax));
    }
    cplx *const o[6] = {out.p[6], out.p[7], out.p[8], out.p[9], out.p[10], out.p[11]};
    zinv_curl5<N, E, Cfg, SG>(bx, by, bz, kx, ky, lds, row, stride, L, t, fft, o, g, i, j0, lmask);
  } else if constexpr (MODE == 6) {
    // velocity gradients: v -> d v_i / d x_j for i, j = 1..3 (out.p[3 i + j],
    // i major), derivk3 (pseudospec3D_hd.f90:22-88) scaled by 1/(nx ny nz)
    const double kx = wavenum(i, g.nx, g.dkx), ky = wavenum(j, g.ny, g.dky);
    const double sc = 1.0 / ((double)g.nx * (double)g.ny * (double)g.nz);
    cplx u[3][E];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int m = 0; m < E; ++m) u[c][m] = load(in.p[c], t + T * m);
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int dir = 0; dir < 3; ++dir) {
        cplx v[E];
#pragma unroll
        for (int m = 0; m < E; ++m) {
          const double kd = dir == 0 ? kx : (dir == 1 ? ky : wavenum(t + T * m, g.nz, g.dkz));
          v[m] = c_scale(c_ik(kd, u[c][m]), sc);
        }
        zinv_emit<N, E, Cfg, SG>(v, lds, row, stride, L, t, fft, out.p[3 * c + dir], g, i, j0, lmask);
      }
  } else if constexpr (MODE == 7) {
    // v -> curl v, rotor3's components formed at each mode
    const double kx = wavenum(i, g.nx, g.dkx), ky = wavenum(j, g.ny, g.dky);
    cplx u[3][E];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int m = 0; m < E; ++m) u[c][m] = load(in.p[c], t + T * m);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      cplx v[E];
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const double kz = wavenum(t + T * m, g.nz, g.dkz);
        v[m] = c == 0 ? c_sub(c_ik(ky, u[2][m]), c_ik(kz, u[1][m]))
               : c == 1 ? c_sub(c_ik(kz, u[0][m]), c_ik(kx, u[2][m]))
                        : c_sub(c_ik(kx, u[1][m]), c_ik(ky, u[0][m]));
      }
      zinv_emit<N, E, Cfg, SG>(v, lds, row, stride, L, t, fft, out.p[c], g, i, j0, lmask);
    }
  } else {
    // MODE 4: (a, b, c, d) -> (a, b, c, grad d).  MODE 5: (v, th) -> (v, curl v, grad th).
    const double kx = wavenum(i, g.nx, g.dkx), ky = wavenum(j, g.ny, g.dky);
    cplx ux[E], uy[E], uz[E];
#pragma unroll
    for (int m = 0; m < E; ++m) {
      ux[m] = load(in.p[0], t + T * m);
      uy[m] = load(in.p[1], t + T * m);
      uz[m] = load(in.p[2], t + T * m);
    }
    if constexpr (MODE == 5) {
      cplx *const o[6] = {out.p[0], out.p[1], out.p[2], out.p[3], out.p[4], out.p[5]};
      zinv_curl5<N, E, Cfg, SG>(ux, uy, uz, kx, ky, lds, row, stride, L, t, fft, o, g, i, j0, lmask);
    } else {
      zinv_emit<N, E, Cfg, SG>(ux, lds, row, stride, L, t, fft, out.p[0], g, i, j0, lmask);
      zinv_emit<N, E, Cfg, SG>(uy, lds, row, stride, L, t, fft, out.p[1], g, i, j0, lmask);
      zinv_emit<N, E, Cfg, SG>(uz, lds, row, stride, L, t, fft, out.p[2], g, i, j0, lmask);
    }
    // derivk3 (pseudospec3D_hd.f90:22-88) of the scalar along x, y, z:
    // Z^-1(i kx d) = i kx Z^-1(d) and likewise for ky, so two transforms
    constexpr int base = MODE == 4 ? 3 : 6;
    cplx d[E];
#pragma unroll
    for (int m = 0; m < E; ++m) d[m] = load(in.p[3], t + T * m);
    {
      cplx w[E];
#pragma unroll
      for (int m = 0; m < E; ++m) w[m] = c_ik(wavenum(t + T * m, g.nz, g.dkz), d[m]);
      zinv_emit<N, E, Cfg, SG>(w, lds, row, stride, L, t, fft, out.p[base + 2], g, i, j0, lmask);
    }
    cplx x[F::SE];
    fft.inv(d, x, row, t);
#pragma unroll
    for (int dir = 0; dir < 2; ++dir) {
      cplx w[F::SE];
      const double kd = dir == 0 ? kx : ky;
      if (F::live(t)) {
#pragma unroll
        for (int m = 0; m < F::SE; ++m) w[m] = c_ik(kd, x[m]);
      }
      zinv_store<N, E, Cfg, SG>(w, lds, row, stride, L, t, out.p[base + dir], g, i, j0, lmask);
    }
  }
}

// Z^-1 with one output field per block (blockIdx.z = member * outputs + field):
// every field of the modes above from its inputs' modes and one transform.
// For launches too small to fill the GPU, where the fields that a block works
// through one after another are what a pass takes: 3 loads, 6 transforms and 6
// tile stores in turn are 12 us at 32^3 to 64^3 whatever the tile, and one of
// each is half of that.  Inputs are read again by each block that needs them
// (cache hits at these sizes), and a curl costs a transform more.
// What output o of a mode is: component c of the fields from f (kind 0 the
// field itself, 1 its derivative along c, 2 their curl, 3 the curl of their
// curl).
struct ZOut {
  int kind, f, c;
};
GHX_DEV ZOut zinv_output(int mode, int o) {
  switch (mode) {
  case 1: case 5: return o < 3 ? ZOut{0, o, 0} : o < 6 ? ZOut{2, 0, o - 3} : ZOut{1, 3, o - 6};
  case 2: return o < 3 ? ZOut{0, o, 0} : o < 6 ? ZOut{2, 0, o - 3} : o < 9 ? ZOut{2, 3, o - 6} : ZOut{3, 3, o - 9};
  case 4: return o < 3 ? ZOut{0, o, 0} : ZOut{1, 3, o - 3};
  case 6: return ZOut{1, o / 3, o % 3};
  case 7: return ZOut{2, 0, o};
  default: return ZOut{0, o, 0};
  }
}

template <int N, typename Cfg = FFTCfgMix<N>>
__global__ __launch_bounds__(kTileBound) void k_zinv_one(FieldSet in_, FieldSet out_, int mode, int nout, GridK g,
                                                 const cplx *__restrict__ twt, int prune_, const unsigned *dirty,
                                                 const double *__restrict__ aux) {
  using F = Line<N, Cfg>;
  constexpr int T = F::T, E = F::KE;
  const int prune = prune_input(prune_, dirty);
  extern __shared__ cplx lds[];
  const int L = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  const int member = blockIdx.z / nout, o = blockIdx.z - member * nout;
  const ZOut w = zinv_output(mode, o);  // the same for the whole block
  int bx, by;
  xcd_tile(bx, by, prune != 0);
  const int i = by, j0 = bx * L, j = j0 + lt;
  const unsigned lmask = prune ? tile_lines_active(g, i, j0, L) : ~0u;
  if (lmask == 0u) return;  // uniform over the block
  F fft;
  fft.load_inv(twt, t);
  const bool ok = j < g.ny && ((lmask >> lt) & 1u);
  const int stride = lds_line_stride(N);
  cplx *row = lds + lt * stride;
  const size_t sline = ((size_t)i * g.ny + (ok ? j : 0)) * N;
  const double kx = wavenum(i, g.nx, g.dkx), ky = wavenum(ok ? j : 0, g.ny, g.dky);
  // component q of the inputs' wavenumber, q mod 3
  auto kq = [&](int q, int m) { return q == 0 ? kx : q == 1 ? ky : wavenum(t + T * m, g.nz, g.dkz); };
  auto load = [&](cplx (&x)[E], int f) {
    const cplx *p = in_.p[f] + (size_t)member * in_.bstride + sline;
#pragma unroll
    for (int m = 0; m < E; ++m) {
      const int k = t + T * m;
      const bool need = ok && (!prune || kn2_of(g, i, j, k) <= g.kmax);
      const cplx y = p[need ? k : 0];
      x[m] = need ? y : c_make(0.0, 0.0);
    }
  };
  const int c1 = w.c == 2 ? 0 : w.c + 1, c2 = w.c == 0 ? 2 : w.c - 1;  // c + 1, c + 2 mod 3
  cplx v[E];
  load(v, w.kind >= 2 ? w.f + c2 : w.f);
  if (w.kind == 1) {
    const double sc = mode == 6 ? 1.0 / ((double)g.nx * (double)g.ny * (double)g.nz) : 1.0;
#pragma unroll
    for (int m = 0; m < E; ++m) v[m] = c_scale(c_ik(kq(w.c, m), v[m]), sc);
  } else if (w.kind >= 2) {
    cplx x[E];
    load(x, w.f + c1);
    if (w.kind == 2) {  // i k_{c+1} a_{c+2} - i k_{c+2} a_{c+1}
#pragma unroll
      for (int m = 0; m < E; ++m) v[m] = c_sub(c_ik(kq(c1, m), v[m]), c_ik(kq(c2, m), x[m]));
    } else {  // the same of b = curl a
      cplx y[E];
      load(y, w.f + w.c);
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const double k0 = kq(w.c, m), k1 = kq(c1, m), k2 = kq(c2, m);
        const cplx b2 = c_sub(c_ik(k0, x[m]), c_ik(k1, y[m])), b1 = c_sub(c_ik(k2, y[m]), c_ik(k0, v[m]));
        v[m] = c_sub(c_ik(k1, b2), c_ik(k2, b1));
      }
    }
  }
  if (mode == 3) {
    const double sxy = aux[i] * aux[g.nxh + (ok ? j : 0)];
#pragma unroll
    for (int m = 0; m < E; ++m) v[m] = c_scale(v[m], sxy * aux[g.nxh + g.ny + t + T * m]);
  }
  zinv_emit<N, E, Cfg>(v, lds, row, stride, L, t, fft, out_.p[o] + (size_t)member * out_.bstride, g, i, j0, lmask);
}

// ---------------------------------------------------------------------------
// Z forward: Q -> S.  Block = (kx index i, ky chunk).  Transposed load.
// ---------------------------------------------------------------------------
template <int N, int E, typename Cfg = FFTCfgMix<N>>
GHX_DEV void zfwd_load(cplx (&v)[E], cplx *lds, cplx *row, int stride, int L, int t, const Line<N, Cfg> &fft,
                       const cplx *src, const GridK &g, int i, int j0, unsigned lmask = ~0u) {
  tile_load_q<E>(lds, stride, L, src, (size_t)g.nxh * g.ny, (size_t)i * g.ny, j0, g.ny, lmask);
  __syncthreads();
  cplx x[Line<N, Cfg>::SE];
  fft.get(x, row, t);
  __syncthreads();
  fft.fwd(x, v, row, t);
}

// prune: only the kept modes of the output are wanted (the caller reads no
// other), so only the dealias disc's lines are loaded (the y forward wrote no
// others) and only their kept modes are written; the rest of `out` keeps
// whatever it held.
template <int N, typename Cfg = FFTCfgMix<N>>
__global__ __launch_bounds__(kTileBound) void k_zfwd(FieldSet in, FieldSet out, int nf, GridK g, const cplx *__restrict__ twt,
                                             int prune) {
  using F = Line<N, Cfg>;
  constexpr int T = F::T, E = F::KE;
  extern __shared__ cplx lds[];
  const int L = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  F fft;  // with this lane's stage roots, loaded once
  fft.load_fwd(twt, t);
  int bx, by;
  xcd_tile(bx, by, prune != 0);
  const int i = by, j0 = bx * L, j = j0 + lt;
  const unsigned lmask = prune ? tile_lines_active(g, i, j0, L) : ~0u;
  if (lmask == 0u) return;  // uniform over the block
  const bool ok = j < g.ny && ((lmask >> lt) & 1u);
  const int stride = lds_line_stride(N);
  cplx *row = lds + lt * stride;
  const size_t sline = ((size_t)i * g.ny + (ok ? j : 0)) * N;
  for (int f = 0; f < nf; ++f) {
    cplx v[E];
    zfwd_load<N, E, Cfg>(v, lds, row, stride, L, t, fft, in.p[f], g, i, j0, lmask);
    if (ok) {
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const int k = t + T * m;
        if (!prune || kn2_of(g, i, j, k) <= g.kmax) out.p[f][sline + k] = v[m];
      }
    }
    __syncthreads();
  }
}

// Projection of pseudospec3D_hd.f90:399-509 (nonlhd3) for one mode.
GHX_DEV void project_hd(const cplx &a, const cplx &b, const cplx &c, double kx, double ky, double kz,
                        double kk2, int i, int j, int k, cplx &gx, cplx &gy, cplx &gz) {
  cplx dot = c_add(c_add(c_scale(a, kx), c_scale(b, ky)), c_scale(c, kz));
  gx = i == 0 ? c_make(-a.x, -a.y) : c_add(c_make(-a.x, -a.y), c_make(kx * dot.x / kk2, kx * dot.y / kk2));
  gy = j == 0 ? c_make(-b.x, -b.y) : c_add(c_make(-b.x, -b.y), c_make(ky * dot.x / kk2, ky * dot.y / kk2));
  gz = k == 0 ? c_make(-c.x, -c.y) : c_add(c_make(-c.x, -c.y), c_make(kz * dot.x / kk2, kz * dot.y / kk2));
}

// Coriolis force of include/roth_rkstep2.f90:6-14 added to the products
// (a, b) = FFT of (w x u)_x,y before the projection: a - 2 omegaz v_y,
// b + 2 omegaz v_x, with om2 = 2 omegaz.
GHX_DEV void coriolis(cplx &a, cplx &b, const cplx &vx, const cplx &vy, double om2) {
  a = c_make(a.x - om2 * vy.x, a.y - om2 * vy.y);
  b = c_make(b.x + om2 * vx.x, b.y + om2 * vx.y);
}

// RK update of include/hd_rkstep2.f90:12-32 for one component:
// v = C + dt*(nu*(-kk2 v) + N + f)*rmp
GHX_DEV cplx rk_update(cplx cc, cplx vv, cplx nl, cplx ff, double kk2, double nu, double dt, double rmp) {
  double lx = -kk2 * vv.x, ly = -kk2 * vv.y;
  double sx = nu * lx + nl.x + ff.x, sy = nu * ly + nl.y + ff.y;
  return c_make(cc.x + dt * sx * rmp, cc.y + dt * sy * rmp);
}

// ---------------------------------------------------------------------------
// Z forward fused with the projection and the RK update for small launches
// (kSmallLines) and the Boussinesq update, one group of lanes per component: the block is G x L lines x T lanes, group c transforms its
// component's tile and updates that component.  The tiles of all components
// and the lanes' v and C are loaded together at the start, so a block waits
// for memory once, and the transforms run side by side; the projection reads
// the other components' modes from their LDS rows.  On large launches the
// kernels below, which take the components in turn, are faster (HD 110
// against 191 us at 256^3): three groups per line leave one block per CU,
// whose loads, transforms and stores then do not overlap.
// KIND 0: HD (include/hd_rkstep2.f90, roth_rkstep2.f90); 1: MHD, blockIdx.z
// the part (0 velocity from fields 0..2 minus 3..5, 1 vector potential from
// fields 6..8); 2: Boussinesq (include/bouss_rkstep2.f90:1-71), component 3
// the temperature.
// ---------------------------------------------------------------------------
struct ZUpdate {
  double dt, rmp, om2, xmom, xtemp;
  double nu, mu;  // mu: of the vector potential or the temperature
  const cplx *v[6], *c[6], *f[6];
  cplx *out[6];
  const uint8_t *fline;
  size_t bstride;
  const double *nu_b;
};

template <int N, int KIND, typename Cfg = FFTCfgMix<N>>
__global__ __launch_bounds__(zrk_bound(KIND)) void k_zrk(FieldSet in_, GridK g, const cplx *__restrict__ twt,
                                                         ZUpdate rk, int prune) {
  using F = Line<N, Cfg>;
  constexpr int T = F::T, E = F::KE, G = zrk_groups(KIND);
  extern __shared__ cplx lds[];
  const int GL = blockDim.x / G, L = GL / T, lsh = 31 - __builtin_clz((unsigned)L);
  // groups are whole waves except for the shortest lines (GL < 64)
  int c = threadIdx.x / GL;
  if (GL % 64 == 0) c = __builtin_amdgcn_readfirstlane(c);
  const int tid = threadIdx.x - c * GL;
  const int lt = tid / T, t = tid % T;
  int bx, by;
  xcd_tile(bx, by, prune != 0);
  const int i = by, j0 = bx * L, j = j0 + lt;
  const unsigned lmask = prune ? tile_lines_active(g, i, j0, L) : ~0u;
  const bool inside = j < g.ny, on = (lmask >> lt) & 1u, ok = inside && on;
  const int part = KIND == 1 ? (int)blockIdx.z : 0;
  const size_t bo = KIND == 0 ? (size_t)blockIdx.z * rk.bstride : 0;
  const int ci = KIND == 1 ? 3 * part + c : c;  // this group's component of the argument arrays
  cplx *out = rk.out[ci] + bo;
  const size_t sline = ((size_t)i * g.ny + (inside ? j : 0)) * N;
  if (prune == 2 && inside && !on) {
    // the output buffers held something else: lines outside the disc are zeroed
#pragma unroll 1
    for (int m = 0; m < E; ++m) out[sline + t + T * m] = c_make(0.0, 0.0);
  }
  if (lmask == 0u) return;  // uniform over the block
  const int stride = lds_line_stride(N);
  cplx *rows = lds + c * L * stride, *row = rows + lt * stride;
  F fft;
  fft.load_fwd(twt, t);
  // the tile of this component's product
  cplx P[E];
  {
    const size_t qs = (size_t)g.nxh * g.ny, qb = (size_t)i * g.ny + j0;
    const size_t io = KIND == 0 ? (size_t)blockIdx.z * in_.bstride : 0;
    const cplx *a = in_.p[KIND == 1 && part ? 6 + c : c] + io;
    const cplx *b = in_.p[KIND == 1 ? 3 + c : c];  // KIND 1, part 0
    cplx w[E];
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const int idx = tid + q * GL, l = idx & (L - 1);
      const bool need = j0 + l < g.ny && ((lmask >> l) & 1u);
      const size_t o = qb + (size_t)(idx >> lsh) * qs + (need ? l : 0);
      cplx x = a[o];
      if constexpr (KIND == 1) {
        if (part == 0) x = c_sub(x, b[o]);
      }
      w[q] = need ? x : c_make(0.0, 0.0);
    }
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const int idx = tid + q * GL;
      rows[(idx & (L - 1)) * stride + lds_pad(idx >> lsh)] = w[q];
    }
  }
  const double kx = wavenum(i, g.nx, g.dkx), ky = wavenum(inside ? j : 0, g.ny, g.dky);
  const cplx *vp = rk.v[ci] + bo, *cp = rk.c[ci] + bo;
  cplx vv[E], cc[E];
  auto kept = [&](int k) { return ok && kn2_of(g, i, j, k) <= g.kmax; };
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int k = t + T * m;
    const size_t s = sline + (kept(k) ? k : 0);
    vv[m] = vp[s];
    cc[m] = cp[s];  // a second hit in the cache where C is v
  }
  __syncthreads();
  cplx x[F::SE];
  fft.get(x, row, t);
  line_sync<T>();  // a line's row is its own from here on
  fft.fwd(x, P, row, t);
  // the other field that this component's product needs: Coriolis v_y, v_x;
  // buoyancy th; heat current v_z
  if constexpr (KIND != 1) {
    const bool rot = rk.om2 != 0.0;
    const cplx *xp = rk.v[KIND == 2 || c < 2 ? c ^ 1 : 0];
    const double xs = c == 0 ? -rk.om2 : c == 1 ? rk.om2 : KIND == 0 ? 0.0 : c == 2 ? rk.xmom : rk.xtemp;
    if (KIND == 2 || rot) {
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const int k = t + T * m;
        const bool need = kept(k) && (c >= 2 ? KIND == 2 : rot);
        const cplx x = xp[bo + sline + (need ? k : 0)];
        if (need) P[m] = c_make(P[m].x + xs * x.x, P[m].y + xs * x.y);
      }
    }
  }
#pragma unroll
  for (int m = 0; m < E; ++m) row[lds_pad(t + T * m)] = P[m];
  // every lane has loaded what it reads of v before any lane stores (out may
  // be v or C), and the other components' modes are in their rows
  __syncthreads();
  if (!ok) return;
  const double nu = KIND == 0 ? (rk.nu_b ? rk.nu_b[blockIdx.z] : rk.nu) : (KIND == 1 ? part != 0 : c == 3) ? rk.mu : rk.nu;
  const cplx *fp = rk.f[ci];
  if (fp && rk.fline && !rk.fline[(size_t)i * g.ny + j]) fp = nullptr;
  if (fp) fp += bo;
  const cplx *row0 = lds + lt * stride, *row1 = row0 + L * stride, *row2 = row1 + L * stride;
  const double kd = c == 0 ? kx : ky;
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int k = t + T * m;
    const size_t s = sline + k;
    const double kz = wavenum(k, g.nz, g.dkz);
    const double kn2 = kn2_of(g, i, j, k);
    const cplx C = cc[m];
    if (kn2 <= g.kmax && kn2 >= g.tiny) {
      const double kk2 = g.anis ? kk2_of(g, kx, ky, kz) : kn2;
      cplx n;
      if (G == 4 && c == 3) {
        n = P[m];
      } else {
        const cplx a = row0[lds_pad(k)], b = row1[lds_pad(k)], d = row2[lds_pad(k)];
        const cplx dot = c_add(c_add(c_scale(a, kx), c_scale(b, ky)), c_scale(d, kz));
        const double kc = c == 2 ? kz : kd;
        const int plane = c == 0 ? i : c == 1 ? j : k;
        n = c_make(-P[m].x, -P[m].y);
        if (plane != 0) n = c_add(n, c_make(kc * dot.x / kk2, kc * dot.y / kk2));
        // gauge3 is the exact negation of this projection
        if (KIND == 1 && part != 0) n = c_make(-n.x, -n.y);
      }
      cplx ff = c_make(0.0, 0.0);
      if (fp) ff = fp[s];
      c_put<KIND == 0>(out + s, rk_update(C, vv[m], n, ff, kk2, nu, rk.dt, rk.rmp));
    } else if (G == 4 && c == 3 && kn2 < g.tiny) {
      out[s] = C;  // the mean of the temperature is carried
    } else if (prune != 1 || kn2 < g.tiny) {
      // outside the kept modes; the k = 0 mode is written in pruned passes
      // too, since the next substep's inverse reads it from this output
      out[s] = c_make(0.0, 0.0);
    }
  }
}

template <int N, typename Cfg = FFTCfgMix<N>, int PF = 0>
__global__ __launch_bounds__(kTileBound) void k_zfwd_rk_hd(FieldSet in_, GridK g, const cplx *__restrict__ twt, RKParams rk,
                                                   int prune) {
  using F = Line<N, Cfg>;
  constexpr int T = F::T, E = F::KE;
  extern __shared__ cplx lds[];
  const int L = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  F fft;  // with this lane's stage roots, loaded once
  fft.load_fwd(twt, t);
  const FieldView in = batch_view(in_, blockIdx.z);
  if (blockIdx.z && rk.bstride) {
    const size_t o = (size_t)blockIdx.z * rk.bstride;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      rk.v[c] += o;
      rk.c[c] += o;
      rk.out[c] += o;
      if (rk.f[c]) rk.f[c] += o;
    }
  }
  if (rk.nu_b) rk.nu = rk.nu_b[blockIdx.z];
  int bx, by;
  xcd_tile(bx, by, prune != 0);
  const int i = by, j0 = bx * L, j = j0 + lt;
  // prune: all state buffers are dealiased (zero outside the kept modes), so
  // only lines inside the dealias disc are transformed and only kept modes
  // are read and written.
  const unsigned lmask = prune ? tile_lines_active(g, i, j0, L) : ~0u;
  // prune == 2: the output buffers held something else, so the lines outside
  // the dealias disc are zeroed here instead of being known to be zero
  if (prune == 2 && j < g.ny && !((lmask >> lt) & 1u)) {
    const size_t s0 = ((size_t)i * g.ny + j) * N;
#pragma unroll 1
    for (int m = 0; m < E; ++m) {
      rk.out[0][s0 + t + T * m] = c_make(0.0, 0.0);
      rk.out[1][s0 + t + T * m] = c_make(0.0, 0.0);
      rk.out[2][s0 + t + T * m] = c_make(0.0, 0.0);
    }
  }
  if (lmask == 0u) return;  // uniform over the block
  const bool ok = j < g.ny && ((lmask >> lt) & 1u);
  const int stride = lds_line_stride(N);
  cplx *row = lds + lt * stride;
  cplx P[3][E];
  if constexpr (PF) {
    // the next field's tile loads are in flight while this field is transformed
    const size_t qs = (size_t)g.nxh * g.ny, qb = (size_t)i * g.ny;
    cplx w[E];
    tile_fetch_q<E>(w, L, in.p[0], qs, qb, j0, g.ny, lmask);
#pragma unroll
    for (int f = 0; f < 3; ++f) {
      tile_put_q<E>(lds, stride, L, w);
      __syncthreads();
      cplx x[F::SE];
      fft.get(x, row, t);
      __syncthreads();
      if (f < 2) tile_fetch_q<E>(w, L, in.p[f + 1], qs, qb, j0, g.ny, lmask);
      fft.fwd(x, P[f], row, t);
      __syncthreads();
    }
  } else {
#pragma unroll
    for (int f = 0; f < 3; ++f) {
      zfwd_load<N, E, Cfg>(P[f], lds, row, stride, L, t, fft, in.p[f], g, i, j0, lmask);
      __syncthreads();
    }
  }
  if (!ok) return;
  const double kx = wavenum(i, g.nx, g.dkx), ky = wavenum(j, g.ny, g.dky);
  const size_t sline = ((size_t)i * g.ny + j) * N;
  const bool forced = rk.f[0] && (!rk.fline || rk.fline[(size_t)i * g.ny + j]);
  const cplx z = c_make(0.0, 0.0);
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int k = t + T * m;
    const size_t s = sline + k;
    const double kz = wavenum(k, g.nz, g.dkz);
    const double kn2 = kn2_of(g, i, j, k);
    if (kn2 <= g.kmax && kn2 >= g.tiny) {
      const double kk2 = g.anis ? kk2_of(g, kx, ky, kz) : kn2;
      cplx n0, n1, n2;
      if (rk.om2 != 0.0) coriolis(P[0][m], P[1][m], rk.v[0][s], rk.v[1][s], rk.om2);
      project_hd(P[0][m], P[1][m], P[2][m], kx, ky, kz, kk2, i, j, k, n0, n1, n2);
      c_put<true>(&rk.out[0][s], rk_update(rk.c[0][s], rk.v[0][s], n0, forced ? rk.f[0][s] : z, kk2, rk.nu, rk.dt, rk.rmp));
      c_put<true>(&rk.out[1][s], rk_update(rk.c[1][s], rk.v[1][s], n1, forced ? rk.f[1][s] : z, kk2, rk.nu, rk.dt, rk.rmp));
      c_put<true>(&rk.out[2][s], rk_update(rk.c[2][s], rk.v[2][s], n2, forced ? rk.f[2][s] : z, kk2, rk.nu, rk.dt, rk.rmp));
    } else if (prune != 1 || kn2 < g.tiny) {
      // outside the kept modes; the k = 0 mode is written in pruned passes
      // too, since the next substep's inverse reads it from this output
      c_put<true>(&rk.out[0][s], z);
      c_put<true>(&rk.out[1][s], z);
      c_put<true>(&rk.out[2][s], z);
    }
    // keep the loads of one mode from being hoisted over the others (register pressure)
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Boussinesq (include/bouss_rkstep2.f90:1-71): in.p[0..2] = FFT of w x u,
// in.p[3] = FFT of -(u . grad th).  Per kept mode: buoyancy xmom th added to
// the z product, nonlhd3 projection, heat current xtemp v_z added to the
// advection, then the updates of v (nu) and th (kappa).  The k = 0 mode keeps
// the step-start mean of th; v is zero there and outside the dealias set.
template <int N, typename Cfg = FFTCfgMix<N>>
__global__ __launch_bounds__(kTileBound) void k_zfwd_rk_bouss(FieldSet in, GridK g, const cplx *__restrict__ twt,
                                                      BoussRKParams rk, int prune) {
  using F = Line<N, Cfg>;
  constexpr int T = F::T, E = F::KE;
  extern __shared__ cplx lds[];
  const int L = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  F fft;  // with this lane's stage roots, loaded once
  fft.load_fwd(twt, t);
  int bx, by;
  xcd_tile(bx, by, prune != 0);
  const int i = by, j0 = bx * L, j = j0 + lt;
  const unsigned lmask = prune ? tile_lines_active(g, i, j0, L) : ~0u;
  // prune == 2: the output buffers held something else, so the lines outside
  // the dealias disc are zeroed here instead of being known to be zero
  if (prune == 2 && j < g.ny && !((lmask >> lt) & 1u)) {
    const size_t s0 = ((size_t)i * g.ny + j) * N;
#pragma unroll 1
    for (int m = 0; m < E; ++m) {
      rk.out[0][s0 + t + T * m] = c_make(0.0, 0.0);
      rk.out[1][s0 + t + T * m] = c_make(0.0, 0.0);
      rk.out[2][s0 + t + T * m] = c_make(0.0, 0.0);
      rk.out[3][s0 + t + T * m] = c_make(0.0, 0.0);
    }
  }
  if (lmask == 0u) return;  // uniform over the block
  const bool ok = j < g.ny && ((lmask >> lt) & 1u);
  const int stride = lds_line_stride(N);
  cplx *row = lds + lt * stride;
  const double kx = wavenum(i, g.nx, g.dkx), ky = wavenum(j < g.ny ? j : 0, g.ny, g.dky);
  const size_t sline = ((size_t)i * g.ny + (ok ? j : 0)) * N;
  const bool forced = ok && rk.f[0] && (!rk.fline || rk.fline[(size_t)i * g.ny + j]);
  const cplx z = c_make(0.0, 0.0);
  // v_z as the nonlinear term saw it, for the heat current: with ord = 1 the
  // update writes over the input (out == v) before the temperature is done.
  // Kept in LDS past the line tiles (each lane rereads only its own modes).
  cplx *vz_in = lds + L * stride + lt * N;
  {
    cplx P[3][E];
#pragma unroll
    for (int f = 0; f < 3; ++f) {
      zfwd_load<N, E, Cfg>(P[f], lds, row, stride, L, t, fft, in.p[f], g, i, j0, lmask);
      __syncthreads();
    }
    if (ok) {
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const int k = t + T * m;
        const size_t s = sline + k;
        const double kz = wavenum(k, g.nz, g.dkz);
        const double kn2 = kn2_of(g, i, j, k);
        if (kn2 <= g.kmax && kn2 >= g.tiny) {
          const double kk2 = g.anis ? kk2_of(g, kx, ky, kz) : kn2;
          vz_in[k] = rk.v[2][s];
          const cplx th = rk.v[3][s];
          const cplx nzb = c_make(P[2][m].x + rk.xmom * th.x, P[2][m].y + rk.xmom * th.y);
          // rotbouss_rkstep2.f90:6-15: Coriolis on x, y beside the gravity on z
          if (rk.om2 != 0.0) coriolis(P[0][m], P[1][m], rk.v[0][s], rk.v[1][s], rk.om2);
          cplx n0, n1, n2;
          project_hd(P[0][m], P[1][m], nzb, kx, ky, kz, kk2, i, j, k, n0, n1, n2);
          rk.out[0][s] = rk_update(rk.c[0][s], rk.v[0][s], n0, forced ? rk.f[0][s] : z, kk2, rk.nu, rk.dt, rk.rmp);
          rk.out[1][s] = rk_update(rk.c[1][s], rk.v[1][s], n1, forced ? rk.f[1][s] : z, kk2, rk.nu, rk.dt, rk.rmp);
          rk.out[2][s] = rk_update(rk.c[2][s], rk.v[2][s], n2, forced ? rk.f[2][s] : z, kk2, rk.nu, rk.dt, rk.rmp);
        } else if (prune != 1 || kn2 < g.tiny) {
          rk.out[0][s] = z;
          rk.out[1][s] = z;
          rk.out[2][s] = z;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  cplx A[E];
  zfwd_load<N, E, Cfg>(A, lds, row, stride, L, t, fft, in.p[3], g, i, j0, lmask);
  if (!ok) return;
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int k = t + T * m;
    const size_t s = sline + k;
    const double kz = wavenum(k, g.nz, g.dkz);
    const double kn2 = kn2_of(g, i, j, k);
    if (kn2 <= g.kmax && kn2 >= g.tiny) {
      const double kk2 = g.anis ? kk2_of(g, kx, ky, kz) : kn2;
      const cplx vz = vz_in[k];
      const cplx a = c_make(A[m].x + rk.xtemp * vz.x, A[m].y + rk.xtemp * vz.y);
      rk.out[3][s] = rk_update(rk.c[3][s], rk.v[3][s], a, forced && rk.f[3] ? rk.f[3][s] : z, kk2, rk.kappa, rk.dt,
                               rk.rmp);
    } else if (kn2 < g.tiny) {
      rk.out[3][s] = rk.c[3][s];
    } else if (prune != 1) {
      rk.out[3][s] = z;
    }
  }
}

// MHD: nonlin3 (pseudospec3D_mhd.f90:108-227) for the velocity from
// (w x u, j x b) (PART 0) and gauge3 (:230-336) for the potential from u x b
// (PART 1).  The two parts are separate launches so that each keeps its
// fields in registers.
template <int N, int PART, typename Cfg = FFTCfgMix<N>>
__global__ __launch_bounds__(kTileBound) void k_zfwd_rk_mhd(FieldSet in, GridK g, const cplx *__restrict__ twt, MHDRKParams rk,
                                                    int prune) {
  using F = Line<N, Cfg>;
  constexpr int T = F::T, E = F::KE;
  extern __shared__ cplx lds[];
  const int L = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  F fft;  // with this lane's stage roots, loaded once
  fft.load_fwd(twt, t);
  int bx, by;
  xcd_tile(bx, by, prune != 0);
  const int i = by, j0 = bx * L, j = j0 + lt;
  const unsigned lmask = prune ? tile_lines_active(g, i, j0, L) : ~0u;
  // prune == 2: the output buffers held something else, so the lines outside
  // the dealias disc are zeroed here instead of being known to be zero
  if (prune == 2 && j < g.ny && !((lmask >> lt) & 1u)) {
    const size_t s0 = ((size_t)i * g.ny + j) * N;
#pragma unroll 1
    for (int m = 0; m < E; ++m) {
      rk.out[(PART == 0 ? 0 : 3)][s0 + t + T * m] = c_make(0.0, 0.0);
      rk.out[(PART == 0 ? 1 : 4)][s0 + t + T * m] = c_make(0.0, 0.0);
      rk.out[(PART == 0 ? 2 : 5)][s0 + t + T * m] = c_make(0.0, 0.0);
    }
  }
  if (lmask == 0u) return;  // uniform over the block
  const bool ok = j < g.ny && ((lmask >> lt) & 1u);
  const int stride = lds_line_stride(N);
  cplx *row = lds + lt * stride;
  // PART 0, velocity: fields 0..2 = w x u, 3..5 = j x b; nonlin3 needs only
  // the difference of their transforms, D = FFT(w x u - j x b), and the
  // difference is taken on the tiles before one transform.  PART 1, vector
  // potential: fields 6..8 = u x b.  The next field's tiles are in flight
  // while this one is transformed.
  const size_t qs = (size_t)g.nxh * g.ny, qb = (size_t)i * g.ny;
  cplx wa[E], wb[E];
  auto fetch = [&](int f) {
    tile_fetch_q<E>(wa, L, in.p[PART == 0 ? f : 6 + f], qs, qb, j0, g.ny, lmask);
    if constexpr (PART == 0) tile_fetch_q<E>(wb, L, in.p[3 + f], qs, qb, j0, g.ny, lmask);
  };
  cplx D[3][E];
  fetch(0);
#pragma unroll
  for (int f = 0; f < 3; ++f) {
    if constexpr (PART == 0) {
#pragma unroll
      for (int q = 0; q < E; ++q) wa[q] = c_sub(wa[q], wb[q]);
    }
    tile_put_q<E>(lds, stride, L, wa);
    __syncthreads();
    cplx x[F::SE];
    fft.get(x, row, t);
    __syncthreads();
    if (f < 2) fetch(f + 1);
    fft.fwd(x, D[f], row, t);
    __syncthreads();
  }
  if (!ok) return;
  constexpr int c0 = PART == 0 ? 0 : 3;
  const double coef = PART == 0 ? rk.nu : rk.mu;
  const double kx = wavenum(i, g.nx, g.dkx), ky = wavenum(j, g.ny, g.dky);
  const size_t sline = ((size_t)i * g.ny + j) * N;
  const bool forced = rk.f[c0] && (!rk.fline || rk.fline[(size_t)i * g.ny + j]);
  const cplx z = c_make(0.0, 0.0);
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int k = t + T * m;
    const size_t s = sline + k;
    const double kz = wavenum(k, g.nz, g.dkz);
    const double kn2 = kn2_of(g, i, j, k);
    if (kn2 <= g.kmax && kn2 >= g.tiny) {
      const double kk2 = g.anis ? kk2_of(g, kx, ky, kz) : kn2;
      cplx n0, n1, n2;
      // nonlin3 is the nonlhd3 projection of D; gauge3 is its negative
      // applied to u x b (negation is exact, so both match the routines)
      project_hd(D[0][m], D[1][m], D[2][m], kx, ky, kz, kk2, i, j, k, n0, n1, n2);
      auto upd = [&](int c, cplx nl) {
        if constexpr (PART == 1) nl = c_make(-nl.x, -nl.y);
        const cplx ff = forced && rk.f[c0 + c] ? rk.f[c0 + c][s] : z;
        rk.out[c0 + c][s] = rk_update(rk.c[c0 + c][s], rk.v[c0 + c][s], nl, ff, kk2, coef, rk.dt, rk.rmp);
      };
      upd(0, n0);
      upd(1, n1);
      upd(2, n2);
    } else if (prune != 1 || kn2 < g.tiny) {  // the k = 0 mode: as in k_zfwd_rk_hd
      rk.out[c0][s] = z;
      rk.out[c0 + 1][s] = z;
      rk.out[c0 + 2][s] = z;
    }
    __builtin_amdgcn_sched_barrier(0);  // one mode's loads at a time (register pressure)
  }
}

// ---------------------------------------------------------------------------
// Y passes between Q[z][kx][ky] (ky fastest) and P[z][ky][kx] (kx fastest,
// rows of nxp >= nx/2+1 points).  Block = (z, kx chunk kx0..kx0+L-1); the
// ky lines are contiguous in Q and the transpose to or from P goes through
// an LDS tile with L-point (L*16-byte) chunks along kx.  Only kx < kxlim is
// touched (kxlim < nx/2+1 when the fields are dealiased).
// ---------------------------------------------------------------------------
// A y launch split over its fields has parts = nf blocks per tile and member,
// one field each; else parts = 1.  inv divides blockIdx.z by parts without a
// division or a branch ahead of the kernel's other argument reads (exact up to
// 65535 for up to kMaxFields parts).
struct YSplit {
  int parts;
  unsigned inv;
};
// (whole fields where the members' fields would be more blocks than a grid's z
// extent holds: 10923 members of six fields)
constexpr long kGridZ = 65535;
static inline YSplit ysplit(bool split, int nf, int batch) {
  const int parts = split && (long)nf * batch <= kGridZ ? nf : 1;
  return YSplit{parts, (unsigned)(((1ull << 31) + parts - 1) / parts)};
}

template <int N, typename Cfg = FFTCfgMix<N>>
__global__ __launch_bounds__(kTileBound) void k_yinv(FieldSet in_, FieldSet out_, int nf_, YSplit sp, GridK g, int nxp,
                                             const cplx *__restrict__ twt, int kxlim, int prune, const unsigned *dirty) {
  using F = Line<N, Cfg>;
  if (dirty && *dirty != 0u) prune = 0, kxlim = g.nxh;  // (as prune_input)
  constexpr int T = F::T, E = F::KE;
  extern __shared__ cplx lds[];
  const int L = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  F fft;  // with this lane's stage roots, loaded once
  fft.load_inv(twt, t);
  // blockIdx.z: member and, where a launch is split over its fields, the
  // block's field (ysplit)
  const int member = __umulhi(2u * blockIdx.z, sp.inv), f0 = (int)blockIdx.z - member * sp.parts;
  const int nf = sp.parts > 1 ? f0 + 1 : nf_;
  const FieldView in = batch_view(in_, member);
  const FieldView out = batch_view(out_, member);
  int bx, by;
  xcd_tile(bx, by);
  const int z = by, kx0 = bx * L, kx = kx0 + lt;
  if (kx0 >= kxlim) return;  // uniform over the block
  const bool ok = kx < kxlim;
  const int stride = lds_line_stride(N);
  cplx *row = lds + lt * stride;
  // dealiased input: Q holds data only on the lines (kx,ky) of the dealias
  // disc; every lane loads inside its line and a select drops the rest
  auto load = [&](int f, cplx (&v)[E]) {
    const cplx *src = in.p[f] + ((size_t)z * g.nxh + (ok ? kx : 0)) * N;
#pragma unroll
    for (int m = 0; m < E; ++m) {
      const int j = t + T * m;
      const bool need = ok && (!prune || kn2_of(g, kx, j, 0) <= g.kmax);
      const cplx x = src[need ? j : 0];
      v[m] = need ? x : c_make(0.0, 0.0);
    }
  };
  // E <= 8: the next field's line is loaded while this one is transformed;
  // wider schedules have no registers for it and rely on a second block per CU
  constexpr bool prefetch = E <= 8;
  cplx nxt[prefetch ? E : 1];
  if constexpr (prefetch) load(f0, nxt);
  for (int f = f0; f < nf; ++f) {
    cplx v[E];
    if constexpr (prefetch) {
#pragma unroll
      for (int m = 0; m < E; ++m) v[m] = nxt[m];
      if (f + 1 < nf) load(f + 1, nxt);  // the next field's line in flight during this one
    } else {
      load(f, v);
    }
    cplx x[F::SE];
    fft.inv(v, x, row, t);
    F::put(x, row, t);
    __syncthreads();
    tile_store_rows<E, true>(lds, stride, L, out.p[f] + (size_t)z * g.ny * nxp + kx0, (size_t)nxp,
                       [=](int l) { return kx0 + l < kxlim; });
    __syncthreads();
  }
}

template <int N, typename Cfg = FFTCfgMix<N>>
__global__ __launch_bounds__(kTileBound) void k_yfwd(FieldSet in_, FieldSet out_, int nf_, YSplit sp, GridK g, int nxp,
                                             const cplx *__restrict__ twt, int kxlim, int prune) {
  using F = Line<N, Cfg>;
  constexpr int T = F::T, E = F::KE;
  extern __shared__ cplx lds[];
  const int L = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  F fft;  // with this lane's stage roots, loaded once
  fft.load_fwd(twt, t);
  // blockIdx.z: member and, where a launch is split over its fields, the
  // block's field (ysplit)
  const int member = __umulhi(2u * blockIdx.z, sp.inv), f0 = (int)blockIdx.z - member * sp.parts;
  const int nf = sp.parts > 1 ? f0 + 1 : nf_;
  const FieldView in = batch_view(in_, member);
  const FieldView out = batch_view(out_, member);
  int bx, by;
  xcd_tile(bx, by);
  const int z = by, kx0 = bx * L, kx = kx0 + lt;
  if (kx0 >= kxlim) return;  // uniform over the block
  const bool ok = kx < kxlim;
  const int stride = lds_line_stride(N);
  cplx *row = lds + lt * stride;
  // The block's tile of a field: E points per thread (L*N points over L*T
  // threads), loaded into registers with in-tile addresses (columns at or
  // beyond kxlim read column kx0 and are zeroed), so the loads issue back to
  // back and the next field's tile is in flight while this one is transformed.
  auto tload = [&](int f, cplx (&w)[E]) {
    const cplx *src = in.p[f] + (size_t)z * g.ny * nxp;
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const int idx = threadIdx.x + q * blockDim.x;
      const int l = idx % L, p = idx / L;
      const bool inside = kx0 + l < kxlim;
      // a 32-bit offset from the block's uniform base (ny * nxp < 2^31)
      const cplx x = src[p * nxp + kx0 + (inside ? l : 0)];
      w[q] = inside ? x : c_make(0.0, 0.0);
    }
  };
  constexpr bool prefetch = E <= 8;  // as in k_yinv
  cplx nxt[E];
  if constexpr (prefetch) tload(f0, nxt);
  for (int f = f0; f < nf; ++f) {
    if constexpr (!prefetch) tload(f, nxt);
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const int idx = threadIdx.x + q * blockDim.x;
      lds[(idx % L) * stride + lds_pad(idx / L)] = nxt[q];
    }
    __syncthreads();
    if constexpr (prefetch) {
      if (f + 1 < nf) tload(f + 1, nxt);
    }
    cplx v[E], x[F::SE];
    F::get(x, row, t);
    __syncthreads();
    fft.fwd(x, v, row, t);
    if (ok) {
      cplx *dst = out.p[f] + ((size_t)z * g.nxh + kx) * N;
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const int j = t + T * m;
        // dealiased output: only the ky of the dealias disc are used downstream
        if (!prune || kn2_of(g, kx, j, 0) <= g.kmax) c_put<true>(dst + j, v[m]);
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// X passes on contiguous rows: P rows (nx/2+1 points, kx fastest) <-> real
// rows of nx points held as N = nx/2 packed complex points.  A row is one
// line of T <= 64 lanes (one wavefront for nx = 512), so these kernels use
// only wave-level synchronisation.  Block = RPB rows.
// ---------------------------------------------------------------------------

// Twiddles of the x pass held by one lane for the whole kernel: the stage
// roots of the half-length transform and the packing twiddles w^k of the
// real <-> half-complex step (k = t + T m).
template <int N, typename Cfg> struct XTw {
  static constexpr int E = Cfg::E, T = Cfg::T;
  TwCache<N, Cfg> stage;
  cplx pack[E];
  GHX_DEV void load(const cplx *twh, const cplx *twx, int t) {
    stage.load(twh, t);
#pragma unroll
    for (int m = 0; m < E; ++m) pack[m] = twx[t + T * m];
  }
};

// The loads of one P row for X^-1: points k = t + T m and the Nyquist point.
// Every lane loads from inside the row (points at kx >= kxlim read point 0
// and are zeroed by a select), so the loads issue back to back and a caller
// can start the next row's loads before transforming this one.
template <int E> struct XRowIn {
  cplx a[E];
  cplx nyq;
};

template <int N, int E, typename Cfg>
GHX_DEV void xrow_load(XRowIn<E> &r, const cplx *src, int t, int kxlim) {
  constexpr int T = Cfg::T;
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int k = t + T * m;
    r.a[m] = src[k < kxlim ? k : 0];
  }
  r.nyq = src[N < kxlim ? N : 0];
}

// Half-spectrum row -> unnormalised c2r of the row, packed: v[m] holds
// (x[2k], x[2k+1]) * nx for k = t + T m.  GHOST's c2r ignores the imaginary
// parts of the kx = 0 and Nyquist entries.  The mirrored points X[N-k] come
// through the line's LDS buffer (slot N holds the Nyquist point).
template <int N, int E, typename Cfg>
GHX_DEV void xrow_inv(cplx (&v)[E], const XRowIn<E> &r, cplx *buf, int t, const XTw<N, Cfg> &tw, int kxlim) {
  using F = LineFFT<N, +1, Cfg>;
  constexpr int T = F::T;
  cplx a[E];
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int k = t + T * m;
    a[m] = k < kxlim ? r.a[m] : c_make(0.0, 0.0);
    buf[lds_pad(k)] = a[m];
  }
  if (t == 0) buf[lds_pad(N)] = N < kxlim ? r.nyq : c_make(0.0, 0.0);
  line_sync<T>();
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int k = t + T * m;
    cplx A = a[m];
    cplx Bs = buf[lds_pad(N - k)];
    if (k == 0) { A.y = 0.0; Bs.y = 0.0; }
    cplx B = c_conj(Bs);
    cplx Xe = c_add(A, B);
    cplx Xo = c_mul(c_sub(A, B), c_conj(tw.pack[m]));
    v[m] = c_add(Xe, c_make(-Xo.y, Xo.x));
  }
  line_sync<T>();
  F::run(v, buf, t, tw.stage);
}

// Packed real row -> r2c half spectrum, stored to a P row (kx < kxlim only).
template <int N, int E, typename Cfg>
GHX_DEV void xrow_fwd(cplx (&v)[E], cplx *buf, int t, const XTw<N, Cfg> &tw, cplx *dst, int kxlim) {
  using F = LineFFT<N, -1, Cfg>;
  constexpr int T = F::T;
  F::run(v, buf, t, tw.stage);
#pragma unroll
  for (int m = 0; m < E; ++m) buf[lds_pad(t + T * m)] = v[m];
  line_sync<T>();
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int k = t + T * m;
    cplx A = v[m];
    cplx B = c_conj(buf[lds_pad((N - k) % N)]);
    cplx Xe = c_scale(c_add(A, B), 0.5);
    cplx d = c_sub(A, B);
    cplx Xo = c_make(0.5 * d.y, -0.5 * d.x);  // -0.5 i (A - B)
    if (k < kxlim) dst[k] = c_add(Xe, c_mul(tw.pack[m], Xo));
  }
  if (t == 0 && N < kxlim) {
    cplx z0 = v[0];
    dst[N] = c_make(z0.x - z0.y, 0.0);
  }
  line_sync<T>();
}

struct RealSet {
  double *p[kMaxFields];
};

template <int N>
__global__ __launch_bounds__(kRowBound) void k_xinv(FieldSet in, RealSet out, int nf, GridK g, int nxp,
                                             const cplx *__restrict__ twh, const cplx *__restrict__ twx,
                                             int kxlim) {
  using Cfg = FFTCfgLow<N>;
  constexpr int T = Cfg::T, E = Cfg::E;
  extern __shared__ cplx lds[];
  const int rpb = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  const long nrows = (long)g.nz * g.ny;
  const long r = (long)blockIdx.x * rpb + lt;
  const bool ok = r < nrows;
  if constexpr (T <= 64) {
    if (!ok) return;  // only wave-level syncs
  }
  const int lim = ok ? kxlim : 0;
  const size_t off = (size_t)(ok ? r : 0) * nxp;
  cplx *buf = lds + lt * lds_line_stride(N);
  XTw<N, Cfg> tw;
  tw.load(twh, twx, t);
  XRowIn<E> cur, nxt;
  xrow_load<N, E, Cfg>(cur, in.p[0] + off, t, lim);
  for (int f = 0; f < nf; ++f) {
    if (f + 1 < nf) xrow_load<N, E, Cfg>(nxt, in.p[f + 1] + off, t, lim);  // next field in flight
    cplx v[E];
    xrow_inv<N, E, Cfg>(v, cur, buf, t, tw, lim);
    if (ok) {
      cplx *dst = reinterpret_cast<cplx *>(out.p[f] + r * g.nx);
#pragma unroll
      for (int m = 0; m < E; ++m) dst[t + T * m] = v[m];
    }
    line_sync<T>();
    cur = nxt;
  }
}

// X^-1 of three fields written interleaved, out[(row * nx + x) * 3 + f]: the
// layout the tracer gather reads (one 4-point stencil row of all three
// components is 96 contiguous bytes).
template <int N>
__global__ __launch_bounds__(kRowBound) void k_xinv3i(FieldSet in, double *out, GridK g, int nxp,
                                               const cplx *__restrict__ twh, const cplx *__restrict__ twx,
                                               int kxlim) {
  using Cfg = FFTCfgLow<N>;
  constexpr int T = Cfg::T, E = Cfg::E;
  extern __shared__ cplx lds[];
  const int rpb = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  const long nrows = (long)g.nz * g.ny;
  const long r = (long)blockIdx.x * rpb + lt;
  const bool ok = r < nrows;
  if constexpr (T <= 64) {
    if (!ok) return;
  }
  const int lim = ok ? kxlim : 0;
  const size_t off = (size_t)(ok ? r : 0) * nxp;
  cplx *buf = lds + lt * lds_line_stride(N);
  XTw<N, Cfg> tw;
  tw.load(twh, twx, t);
  XRowIn<E> r0, r1;
  xrow_load<N, E, Cfg>(r0, in.p[0] + off, t, lim);
  xrow_load<N, E, Cfg>(r1, in.p[1] + off, t, lim);
  cplx v[3][E];
  xrow_inv<N, E, Cfg>(v[0], r0, buf, t, tw, lim);
  xrow_load<N, E, Cfg>(r0, in.p[2] + off, t, lim);
  xrow_inv<N, E, Cfg>(v[1], r1, buf, t, tw, lim);
  xrow_inv<N, E, Cfg>(v[2], r0, buf, t, tw, lim);
  if (!ok) return;
  // lane point k holds x = 2k and 2k+1: six consecutive doubles, 16-byte aligned
  double2 *dst = reinterpret_cast<double2 *>(out + (size_t)r * g.nx * 3);
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int k = t + T * m;
    dst[3 * k + 0] = make_double2(v[0][m].x, v[1][m].x);
    dst[3 * k + 1] = make_double2(v[2][m].x, v[0][m].y);
    dst[3 * k + 2] = make_double2(v[1][m].y, v[2][m].y);
  }
}

template <int N>
__global__ __launch_bounds__(kRowBound) void k_xfwd(RealSet in, FieldSet out, int nf, GridK g, int nxp,
                                             const cplx *__restrict__ twh, const cplx *__restrict__ twx) {
  using Cfg = FFTCfgLow<N>;
  constexpr int T = Cfg::T, E = Cfg::E;
  extern __shared__ cplx lds[];
  const int rpb = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  const long nrows = (long)g.nz * g.ny;
  const long r = (long)blockIdx.x * rpb + lt;
  const bool ok = r < nrows;
  if constexpr (T <= 64) {
    if (!ok) return;
  }
  cplx *buf = lds + lt * lds_line_stride(N);
  XTw<N, Cfg> tw;
  tw.load(twh, twx, t);
  const size_t roff = (size_t)(ok ? r : 0) * g.nx;
  cplx cur[E], nxt[E];
  {
    const cplx *src = reinterpret_cast<const cplx *>(in.p[0] + roff);
#pragma unroll
    for (int m = 0; m < E; ++m) cur[m] = src[t + T * m];
  }
  for (int f = 0; f < nf; ++f) {
    if (f + 1 < nf) {
      const cplx *src = reinterpret_cast<const cplx *>(in.p[f + 1] + roff);
#pragma unroll
      for (int m = 0; m < E; ++m) nxt[m] = src[t + T * m];
    }
    cplx v[E];
#pragma unroll
    for (int m = 0; m < E; ++m) v[m] = ok ? cur[m] : c_make(0.0, 0.0);
    xrow_fwd<N, E, Cfg>(v, buf, t, tw, out.p[f] + (ok ? r : 0) * nxp, ok ? g.nxh : 0);
#pragma unroll
    for (int m = 0; m < E; ++m) cur[m] = nxt[m];
  }
}

// ---------------------------------------------------------------------------
// Two-for-one x passes.  Two Hermitian half rows A, B (kx = 0..NX/2) make one
// complex line of NX points, z[k] = A[k] + i B[k] with A[NX-k] = conj A[k];
// its inverse transform is x_a + i x_b, the two real rows at once.  Forward,
// z = x_a + i x_b gives A[k] = (Z[k] + conj Z[NX-k])/2 and
// B[k] = (Z[k] - conj Z[NX-k])/(2i).  Against one half-length transform per
// row plus its packing step, a pair costs one full-length transform (two LDS
// exchanges for NX = 512 with radix 8^3) and no mirror exchange on the
// inverse side: the mirrored points are read from the row itself.
// ---------------------------------------------------------------------------
// Loads of one pair: lane t takes the points k = t + T m of the full line,
// the upper half from the mirrored kx.  Points with kx >= kxlim read kx = 0
// (kept in-row so the loads issue back to back) and are zeroed when the line
// is formed.
template <int NX, int E, int T>
GHX_DEV void xpair_load(cplx (&A)[E], cplx (&B)[E], const cplx *sa, const cplx *sb, int t, int kxlim) {
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int k = t + T * m;
    const int kk = k <= NX / 2 ? k : NX - k;
    const int i = kk < kxlim ? kk : 0;
    A[m] = sa[i];
    B[m] = sb[i];
  }
}

// z[m] = A[k] + i B[k] over the full line.  GHOST's c2r ignores the
// imaginary parts of the kx = 0 and Nyquist entries.
// With hasb false the line carries A alone (B taken as zero).
template <int NX, int E, int T>
GHX_DEV void xpair_make(cplx (&z)[E], const cplx (&A)[E], const cplx (&B)[E], int t, int kxlim, bool hasb = true) {
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int k = t + T * m;
    const int kk = k <= NX / 2 ? k : NX - k;
    const bool live = kk < kxlim;
    const bool realpt = (kk == 0) || (kk == NX / 2);
    const double s = k > NX / 2 ? -1.0 : 1.0;  // upper half: conjugate
    const bool lb = live && hasb;
    const double ar = live ? A[m].x : 0.0, br = lb ? B[m].x : 0.0;
    const double ai = (live && !realpt) ? s * A[m].y : 0.0, bi = (lb && !realpt) ? s * B[m].y : 0.0;
    z[m] = c_make(ar - bi, ai + br);
  }
}

// Two rows of one field in one line, each at its own scale.  A row transformed
// alone has a rounding error relative to itself; in a line with a larger one it
// would take the larger one's, and a zero row would come out as noise.  So both
// are brought to order one by powers of two (exact) before they are combined,
// and back after the transform (RowScale::out).  A zero row comes out zero; a
// row that holds Inf or NaN is left out of the line and comes out NaN.
struct RowScale {
  double in, out;
};
// exponent of the row's largest component, times two, with the lowest bit set
// unless the row is zero
template <int E> GHX_DEV unsigned row_key(const cplx (&A)[E]) {
  unsigned hi = 0, lo = 0;
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const unsigned long long x = __builtin_bit_cast(unsigned long long, A[m].x);
    const unsigned long long y = __builtin_bit_cast(unsigned long long, A[m].y);
    const unsigned hx = (unsigned)(x >> 32) & 0x7fffffffu, hy = (unsigned)(y >> 32) & 0x7fffffffu;
    hi = hi > hx ? hi : hx;
    hi = hi > hy ? hi : hy;
    lo |= (unsigned)x | (unsigned)y;
  }
  return (hi >> 20) * 2u + ((hi | lo) != 0u ? 1u : 0u);
}
GHX_DEV RowScale row_scale(unsigned key) {
  unsigned e = key >> 1;
  if (e == 2047u) return RowScale{0.0, __builtin_nan("")};
  if (key == 0u) return RowScale{0.0, 0.0};
  e = e < 1u ? 1u : e > 2045u ? 2045u : e;
  return RowScale{__builtin_bit_cast(double, (unsigned long long)(2046u - e) << 52),
                  __builtin_bit_cast(double, (unsigned long long)e << 52)};
}
// z = A sa.in + i B sb.in, A and B masked as in xpair_make
template <int NX, int E, int T>
GHX_DEV void xpair_make_scaled(cplx (&z)[E], cplx (&A)[E], cplx (&B)[E], int t, int kxlim, bool hasb, RowScale &sa,
                               RowScale &sb) {
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int k = t + T * m;
    const int kk = k <= NX / 2 ? k : NX - k;
    const bool live = kk < kxlim, lb = live && hasb;
    const bool realpt = (kk == 0) || (kk == NX / 2);
    const double s = k > NX / 2 ? -1.0 : 1.0;  // upper half: conjugate
    A[m] = c_make(live ? A[m].x : 0.0, live && !realpt ? s * A[m].y : 0.0);
    B[m] = c_make(lb ? B[m].x : 0.0, lb && !realpt ? s * B[m].y : 0.0);
  }
  typedef unsigned short us2 __attribute__((ext_vector_type(2)));
  us2 key = {(unsigned short)row_key<E>(A), (unsigned short)row_key<E>(B)};
#pragma unroll
  for (int o = T / 2; o > 0; o >>= 1)
    key = __builtin_elementwise_max(key, __builtin_bit_cast(us2, __shfl_xor(__builtin_bit_cast(int, key), o, 64)));
  sa = row_scale(key.x);
  sb = row_scale(key.y);
  if ((key.x >> 1) == 2047u || (key.y >> 1) == 2047u) {
#pragma unroll
    for (int m = 0; m < E; ++m) {
      if ((key.x >> 1) == 2047u) A[m] = c_make(0.0, 0.0);
      if ((key.y >> 1) == 2047u) B[m] = c_make(0.0, 0.0);
    }
  }
#pragma unroll
  for (int m = 0; m < E; ++m) z[m] = c_make(A[m].x * sa.in - B[m].y * sb.in, A[m].y * sa.in + B[m].x * sb.in);
}

// Z = forward transform of x_a + i x_b in natural order (z[m] = Z[t + T m]);
// stores A[k], B[k] for k < kxlim (k <= NX/2) to the rows da, db.  The
// mirrored Z[NX-k] come through the line's LDS buffer.
template <int NX, int E, int T>
GHX_DEV void xpair_store2(const cplx (&z)[E], cplx *buf, int t, cplx *da, cplx *db, int kxlim) {
#pragma unroll
  for (int m = 0; m < E; ++m) buf[lds_pad(t + T * m)] = z[m];
  line_sync<T>();
#pragma unroll
  for (int m = 0; m <= E / 2; ++m) {
    const int k = t + T * m;
    if (k <= NX / 2) {
      const cplx Zc = c_conj(buf[lds_pad((NX - k) % NX)]);
      const cplx a = c_scale(c_add(z[m], Zc), 0.5);
      const cplx d = c_sub(z[m], Zc);
      const cplx b = c_make(0.5 * d.y, -0.5 * d.x);  // -0.5 i (Z - conj Z')
      if (k < kxlim) {
        da[k] = a;
        db[k] = b;
      }
    }
  }
  line_sync<T>();
}

// single row: z = forward transform of x_a (imaginary input zero) is A itself
template <int NX, int E, int T>
GHX_DEV void xpair_store1(const cplx (&z)[E], int t, cplx *da, int kxlim) {
#pragma unroll
  for (int m = 0; m <= E / 2; ++m) {
    const int k = t + T * m;
    if (k <= NX / 2 && k < kxlim) da[k] = z[m];
  }
}

// x_a + i x_b -> the line's samples n = t + T m; the single-row form leaves
// the imaginary input zero
template <int E>
GHX_DEV void xpair_real(cplx (&z)[E], const double *sa, const double *sb, int t, int T) {
#pragma unroll
  for (int m = 0; m < E; ++m) z[m] = c_make(sa[t + T * m], sb ? sb[t + T * m] : 0.0);
}

// X^-1 of nf fields, two rows per transform (the last of an odd count alone).
template <int NX>
__global__ __launch_bounds__(kRowBound) void k_xinv2(FieldSet in, RealSet out, int nf, GridK g, int nxp,
                                              const cplx *__restrict__ twt, int kxlim) {
  using X = Line<NX, FFTCfgMix<NX>>;
  static_assert(X::T <= 64, "one row per wavefront or less");
  constexpr int T = X::T, A = X::A, KE = X::KE, SE = X::SE;
  extern __shared__ cplx lds[];
  const int rpb = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  const long r = (long)blockIdx.x * rpb + lt;
  if (r >= (long)g.nz * g.ny) return;
  const size_t off = (size_t)r * nxp, roff = (size_t)r * NX;
  cplx *buf = lds + lt * lds_line_stride(NX);
  X fft;
  fft.load_inv(twt, t);
  cplx a[KE], b[KE], z[KE], x[SE];
  const int np = (nf + 1) / 2, last = nf - 1;
  xpair_load<NX, KE, T>(a, b, in.p[0] + off, in.p[last ? 1 : 0] + off, t, kxlim);
  for (int p = 0; p < np; ++p) {
    const bool two = 2 * p < last;
    xpair_make<NX, KE, T>(z, a, b, t, kxlim, two);
    if (p + 1 < np) {  // next pair in flight
      const int fa = 2 * p + 2;
      xpair_load<NX, KE, T>(a, b, in.p[fa] + off, in.p[fa < last ? fa + 1 : fa] + off, t, kxlim);
    }
    fft.inv(z, x, buf, t);
    if (X::live(t)) {
      double *da = out.p[2 * p] + roff;
#pragma unroll
      for (int m = 0; m < SE; ++m) da[t + A * m] = x[m].x;
      if (two) {
        double *db = out.p[2 * p + 1] + roff;
#pragma unroll
        for (int m = 0; m < SE; ++m) db[t + A * m] = x[m].y;
      }
    }
  }
}

// A lone field's rows, paired with each other: rows 2p and 2p + 1 make one
// complex line, half a transform per row; alone, with a zero imaginary part, a
// row costs a whole one.  One field, alone against paired: x inverse 519 -> 389
// us at 512^3, 70 -> 53 at 256^3, 429 -> 203 at 384^3, 55 -> 30 at 192^3 (6-point
// schedule); x forward 390 -> 192 at 384^3, 42 -> 25 at 192^3, 10.7 -> 10.3 at
// 128^3, but 49 -> 52 at 256^3 and 397 -> 421 at 512^3, which keep the lone form
// (pair_rows_fwd).  The last of an odd count stays in its launch: as one of its
// own 26.1 against 24.6 us for three inverses at 128^3, 79 against 74 at 192^3,
// 565 against 563 at 512 x 512 x 256.  The last row of an odd count goes alone.
// The inverse brings each row to its own scale (xpair_make_scaled) and reads
// two roots per radix-8 stage, since a row alone drops the imaginary half of
// its rounding error: c2r alone | paired with one root | as here, 1e-16: 4.63 |
// 4.94 | 4.54 at 128^3, 4.14 | 4.62 | 3.88 at 512 x 64 x 32.  Neither shows in
// the times (c2r of 512^3 1157 -> 1156 us); reading every power does (1180).
constexpr bool pair_rows_fwd(int nx) { return nx % 3 == 0 || nx <= 128; }
template <int NX>
__global__ __launch_bounds__(kRowBound) void k_xinv_rows(const cplx *__restrict__ in, double *__restrict__ out,
                                                         long nrows, int nxp, const cplx *__restrict__ twt,
                                                         int kxlim) {
  using X = Line<NX, FFTCfgRoots<FFTCfgMix<NX>, false>>;
  static_assert(X::T <= 64, "one row per wavefront or less");
  constexpr int T = X::T, A = X::A, KE = X::KE, SE = X::SE;
  extern __shared__ cplx lds[];
  const int rpb = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  const long r = 2 * ((long)blockIdx.x * rpb + lt);
  if (r >= nrows) return;
  const bool two = r + 1 < nrows;
  cplx *buf = lds + lt * lds_line_stride(NX);
  X fft;
  fft.load_inv(twt, t);
  const cplx *sa = in + (size_t)r * nxp;
  cplx a[KE], b[KE], z[KE], x[SE];
  xpair_load<NX, KE, T>(a, b, sa, two ? sa + nxp : sa, t, kxlim);
  RowScale ra, rb;
  xpair_make_scaled<NX, KE, T>(z, a, b, t, kxlim, two, ra, rb);
  fft.inv(z, x, buf, t);
  if (!X::live(t)) return;
  double *da = out + (size_t)r * NX;
#pragma unroll
  for (int m = 0; m < SE; ++m) da[t + A * m] = x[m].x * ra.out;
  if (two) {
#pragma unroll
    for (int m = 0; m < SE; ++m) da[NX + t + A * m] = x[m].y * rb.out;
  }
}
template <int NX>
__global__ __launch_bounds__(kRowBound) void k_xfwd_rows(const double *__restrict__ in, cplx *__restrict__ out,
                                                         long nrows, int nxp, const cplx *__restrict__ twt) {
  using X = Line<NX, FFTCfgMix<NX>>;
  static_assert(X::T <= 64, "one row per wavefront or less");
  constexpr int T = X::T, A = X::A, KE = X::KE, SE = X::SE;
  extern __shared__ cplx lds[];
  const int rpb = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  const long r = 2 * ((long)blockIdx.x * rpb + lt);
  if (r >= nrows) return;
  const bool two = r + 1 < nrows;
  cplx *buf = lds + lt * lds_line_stride(NX);
  X fft;
  fft.load_fwd(twt, t);
  const double *sa = in + (size_t)r * NX;
  cplx x[SE], z[KE];
  if (X::live(t)) xpair_real<SE>(x, sa, two ? sa + NX : nullptr, t, A);
  fft.fwd(x, z, buf, t);
  cplx *da = out + (size_t)r * nxp;
  if (two) xpair_store2<NX, KE, T>(z, buf, t, da, da + nxp, NX / 2 + 1);
  else xpair_store1<NX, KE, T>(z, t, da, NX / 2 + 1);
}

// X^-1 of three fields written interleaved (the tracer layout of k_xinv3i),
// pairs (0, 1) and (2, alone).
template <int NX>
__global__ __launch_bounds__(kRowBound) void k_xinv3i2(FieldSet in, double *out, GridK g, int nxp,
                                                const cplx *__restrict__ twt, int kxlim) {
  using X = Line<NX, FFTCfgMix<NX>>;
  static_assert(X::T <= 64, "one row per wavefront or less");
  constexpr int T = X::T, A = X::A, KE = X::KE, SE = X::SE;
  extern __shared__ cplx lds[];
  const int rpb = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  const long r = (long)blockIdx.x * rpb + lt;
  if (r >= (long)g.nz * g.ny) return;
  const size_t off = (size_t)r * nxp;
  cplx *buf = lds + lt * lds_line_stride(NX);
  X fft;
  fft.load_inv(twt, t);
  cplx a[KE], b[KE], z[KE], z0[SE], z1[SE];
  xpair_load<NX, KE, T>(a, b, in.p[0] + off, in.p[1] + off, t, kxlim);
  xpair_make<NX, KE, T>(z, a, b, t, kxlim);
  xpair_load<NX, KE, T>(a, b, in.p[2] + off, in.p[2] + off, t, kxlim);
  fft.inv(z, z0, buf, t);
  xpair_make<NX, KE, T>(z, a, b, t, kxlim, false);
  fft.inv(z, z1, buf, t);
  if (!X::live(t)) return;
  double *dst = out + (size_t)r * NX * 3;
#pragma unroll
  for (int m = 0; m < SE; ++m) {
    const int n = t + A * m;
    d_put<true>(dst + 3 * n + 0, z0[m].x);
    d_put<true>(dst + 3 * n + 1, z0[m].y);
    d_put<true>(dst + 3 * n + 2, z1[m].x);
  }
}

// X^-1 of three fields, kept only as the largest squared norm of the points a
// block sees (maxabs): the three real fields are neither written nor read back.
// Rows in a grid-stride loop, the next row's first pair loaded ahead.  At 256^3
// 125 us for what took 141 (x inverse) and 101 us (norms of the real fields).
template <int NX>
__global__ __launch_bounds__(kRowBound) void k_xnorm2(FieldSet in, double *part, GridK g, int nxp,
                                                      const cplx *__restrict__ twt, int kxlim) {
  using X = Line<NX, FFTCfgMix<NX>>;
  static_assert(X::T <= 64, "one row per wavefront or less");
  constexpr int T = X::T, KE = X::KE, SE = X::SE;
  extern __shared__ cplx lds[];
  __shared__ double best[kRowBound / 64];
  const int rpb = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  const long nrows = (long)g.nz * g.ny, hop = (long)gridDim.x * rpb;
  cplx *buf = lds + lt * lds_line_stride(NX);
  X fft;
  fft.load_inv(twt, t);
  double big = 0.0;
  long r = (long)blockIdx.x * rpb + lt;
  if (r < nrows) {  // whole lines only: wave-level syncs inside
    cplx a[KE], b[KE], z[KE], z0[SE], z1[SE];
    xpair_load<NX, KE, T>(a, b, in.p[0] + (size_t)r * nxp, in.p[1] + (size_t)r * nxp, t, kxlim);
    for (; r < nrows; r += hop) {
      const size_t off = (size_t)r * nxp;
      xpair_make<NX, KE, T>(z, a, b, t, kxlim);
      xpair_load<NX, KE, T>(a, b, in.p[2] + off, in.p[2] + off, t, kxlim);
      fft.inv(z, z0, buf, t);
      xpair_make<NX, KE, T>(z, a, b, t, kxlim, false);
      if (r + hop < nrows) {
        const size_t no = (size_t)(r + hop) * nxp;
        xpair_load<NX, KE, T>(a, b, in.p[0] + no, in.p[1] + no, t, kxlim);
      }
      fft.inv(z, z1, buf, t);
      if (X::live(t)) {
#pragma unroll
        for (int m = 0; m < SE; ++m)
          big = fmax(big, z0[m].x * z0[m].x + z0[m].y * z0[m].y + z1[m].x * z1[m].x);
      }
    }
  }
  // (kRowBound lanes are whole waves; a narrower block leaves its missing lanes out)
  for (int o = 32; o > 0; o >>= 1) big = fmax(big, __shfl_xor(big, o, 64));
  if (threadIdx.x % 64 == 0) best[threadIdx.x / 64] = big;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 1; q < (int)(blockDim.x + 63) / 64; ++q) big = fmax(big, best[q]);
    part[blockIdx.x] = big;
  }
}

// X of nf real rows, two rows per transform.
template <int NX>
__global__ __launch_bounds__(kRowBound) void k_xfwd2(RealSet in, FieldSet out, int nf, GridK g, int nxp,
                                              const cplx *__restrict__ twt) {
  using X = Line<NX, FFTCfgMix<NX>>;
  static_assert(X::T <= 64, "one row per wavefront or less");
  constexpr int T = X::T, A = X::A, KE = X::KE, SE = X::SE;
  extern __shared__ cplx lds[];
  const int rpb = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  const long r = (long)blockIdx.x * rpb + lt;
  if (r >= (long)g.nz * g.ny) return;
  const size_t off = (size_t)r * nxp, roff = (size_t)r * NX;
  cplx *buf = lds + lt * lds_line_stride(NX);
  X fft;
  fft.load_fwd(twt, t);
  cplx x[SE], nxt[SE], z[KE];
  const int np = (nf + 1) / 2;
  if (X::live(t)) xpair_real<SE>(x, in.p[0] + roff, nf > 1 ? in.p[1] + roff : nullptr, t, A);
  for (int p = 0; p < np; ++p) {
    const bool two = 2 * p + 1 < nf;
    if (p + 1 < np) {
      const int fa = 2 * p + 2;
      if (X::live(t)) xpair_real<SE>(nxt, in.p[fa] + roff, fa + 1 < nf ? in.p[fa + 1] + roff : nullptr, t, A);
    }
    fft.fwd(x, z, buf, t);
    if (two)
      xpair_store2<NX, KE, T>(z, buf, t, out.p[2 * p] + off, out.p[2 * p + 1] + off, NX / 2 + 1);
    else
      xpair_store1<NX, KE, T>(z, t, out.p[2 * p] + off, NX / 2 + 1);
#pragma unroll
    for (int m = 0; m < SE; ++m) x[m] = nxt[m];
  }
}

// Fused X^-1 . ((A_x B_x + A_y B_y) + A_z B_z) tmp . X (advect3) with pairs
// (A_x, A_y), (A_z, B_x), (B_y, B_z); fields as k_xdot.
template <int NX>
__global__ __launch_bounds__(kRowBound) void k_xdot2(FieldSet in, FieldSet out, GridK g, int nxp,
                                              const cplx *__restrict__ twt, int kxin, int kxout, const unsigned *dirty) {
  const int kxlim = dirty && *dirty != 0u ? g.nxh : kxin;  // (as prune_input)
  using X = Line<NX, FFTCfgMix<NX>>;
  static_assert(X::T <= 64, "one row per wavefront or less");
  constexpr int T = X::T, KE = X::KE, SE = X::SE;
  extern __shared__ cplx lds[];
  const int rpb = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  const long r = (long)blockIdx.x * rpb + lt;
  if (r >= (long)g.nz * g.ny) return;
  const size_t off = (size_t)r * nxp;
  cplx *buf = lds + lt * lds_line_stride(NX);
  const double tmp = -g.inv_n6;
  X fft;
  fft.load_inv(twt, t);
  cplx a[KE], b[KE], z[KE], z0[SE], z1[SE], z2[SE];
  xpair_load<NX, KE, T>(a, b, in.p[0] + off, in.p[1] + off, t, kxlim);
  xpair_make<NX, KE, T>(z, a, b, t, kxlim);
  xpair_load<NX, KE, T>(a, b, in.p[2] + off, in.p[3] + off, t, kxlim);
  fft.inv(z, z0, buf, t);
  xpair_make<NX, KE, T>(z, a, b, t, kxlim);
  xpair_load<NX, KE, T>(a, b, in.p[4] + off, in.p[5] + off, t, kxlim);
  fft.inv(z, z1, buf, t);
  xpair_make<NX, KE, T>(z, a, b, t, kxlim);
  fft.inv(z, z2, buf, t);
  // samples: A_x = z0.x, A_y = z0.y, A_z = z1.x, B_x = z1.y, B_y = z2.x, B_z = z2.y
  fft.load_fwd_too(twt, t);
  if (X::live(t)) {
#pragma unroll
    for (int m = 0; m < SE; ++m)
      z0[m] = c_make(((z0[m].x * z1[m].y + z0[m].y * z2[m].x) + z1[m].x * z2[m].y) * tmp, 0.0);
  }
  fft.fwd(z0, z, buf, t);
  xpair_store1<NX, KE, T>(z, t, out.p[0] + off, kxout);
}

// Fused X^-1 . (P x Q)/N^6 . X with two-for-one transforms: pairs (P_x, P_y),
// (P_z, Q_x), (Q_y, Q_z) inverse, (out_x, out_y) and out_z forward.  Same
// fields, products and operand order as k_xcross.  One row per line of
// T <= 64 lanes.  Two waves per SIMD: a third would put registers of the 3 *
// 2^k rows into scratch, 20 of them and 726 -> 1072 us at 384^3.
template <int NX>
__global__ __launch_bounds__(kRowBound) __attribute__((amdgpu_waves_per_eu(2))) void k_xcross2(FieldSet in_, FieldSet out_, GridK g, int nxp,
                                                const cplx *__restrict__ twt, int kxin, int kxout, const unsigned *dirty) {
  const int kxlim = dirty && *dirty != 0u ? g.nxh : kxin;  // (as prune_input)
  using X = Line<NX, FFTCfgMix<NX>>;
  static_assert(X::T <= 64, "one row per wavefront or less");
  constexpr int T = X::T, KE = X::KE, SE = X::SE;
  extern __shared__ cplx lds[];
  const int rpb = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  const long nrows = (long)g.nz * g.ny;
  const long r = (long)blockIdx.x * rpb + lt;
  if (r >= nrows) return;  // whole lines only: wave-level syncs
  const size_t off = (size_t)r * nxp;
  cplx *buf = lds + lt * lds_line_stride(NX);
  const double tmp = g.inv_n6;
  const FieldView in = batch_view(in_, blockIdx.y);
  const FieldView out = batch_view(out_, blockIdx.y);
  X fft;
  fft.load_inv(twt, t);
  cplx a[KE], b[KE], z[KE], z0[SE], z1[SE], z2[SE];
  xpair_load<NX, KE, T>(a, b, in.p[0] + off, in.p[1] + off, t, kxlim);
  xpair_make<NX, KE, T>(z, a, b, t, kxlim);
  xpair_load<NX, KE, T>(a, b, in.p[2] + off, in.p[3] + off, t, kxlim);
  fft.inv(z, z0, buf, t);
  xpair_make<NX, KE, T>(z, a, b, t, kxlim);
  xpair_load<NX, KE, T>(a, b, in.p[4] + off, in.p[5] + off, t, kxlim);
  fft.inv(z, z1, buf, t);
  xpair_make<NX, KE, T>(z, a, b, t, kxlim);
  fft.inv(z, z2, buf, t);
  // samples: P_x = z0.x, P_y = z0.y, P_z = z1.x, Q_x = z1.y, Q_y = z2.x, Q_z = z2.y
  fft.load_fwd_too(twt, t);
  if (X::live(t)) {
#pragma unroll
    for (int m = 0; m < SE; ++m) {
      const double px = z0[m].x, py = z0[m].y, pz = z1[m].x, qx = z1[m].y, qy = z2[m].x, qz = z2[m].y;
      const double ox = (py * qz - qy * pz) * tmp;
      const double oy = (pz * qx - qz * px) * tmp;
      const double oz = (px * qy - qx * py) * tmp;
      z0[m] = c_make(ox, oy);
      z1[m] = c_make(oz, 0.0);
    }
  }
  fft.fwd(z0, z, buf, t);
  xpair_store2<NX, KE, T>(z, buf, t, out.p[0] + off, out.p[1] + off, kxout);
  fft.fwd(z1, z, buf, t);
  xpair_store1<NX, KE, T>(z, t, out.p[2] + off, kxout);
}

// Fused X^-1 . (P x Q)/N^6 . X on P rows with GHOST's operand order
// (pseudospec3D_hd.f90:377-389): out_x = (P_y Q_z - Q_y P_z) tmp,
// out_y = (P_z Q_x - Q_z P_x) tmp, out_z = (P_x Q_y - Q_x P_y) tmp.
// Fields: in.p[0..2] = P, in.p[3..5] = Q; out.p[0..2].  Only kx < kxlim is
// read and written (dealiased inputs, dealiased use of the outputs).  Each
// row's next input is loaded before the current one is transformed.
template <int N, int W, int SB>
__global__ __launch_bounds__(kRowBound) __attribute__((amdgpu_waves_per_eu(W))) void k_xcross(
    FieldSet in_, FieldSet out_, GridK g, int nxp, const cplx *__restrict__ twh, const cplx *__restrict__ twx,
    int kxin, int kxout, const unsigned *dirty) {
  const int kxlim = dirty && *dirty != 0u ? g.nxh : kxin;  // (as prune_input)
  using Cfg = FFTCfgLow<N>;
  constexpr int T = Cfg::T, E = Cfg::E;
  extern __shared__ cplx lds[];
  const int rpb = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  const long nrows = (long)g.nz * g.ny;
  const long r = (long)blockIdx.x * rpb + lt;
  const bool ok = r < nrows;
  if constexpr (T <= 64) {
    if (!ok) return;
  }
  const int lim = ok ? kxlim : 0, lout = ok ? kxout : 0;
  const size_t off = (size_t)(ok ? r : 0) * nxp;
  cplx *buf = lds + lt * lds_line_stride(N);
  const double tmp = g.inv_n6;
  const FieldView in = batch_view(in_, blockIdx.y);
  const FieldView out = batch_view(out_, blockIdx.y);
  XTw<N, Cfg> tw;
  tw.load(twh, twx, t);
  cplx qx[E], qy[E], qz[E], ay[E], az[E];
  XRowIn<E> ra, rb;
#define GHX_PHASE() do { if constexpr (SB) __builtin_amdgcn_sched_barrier(0); } while (0)
  xrow_load<N, E, Cfg>(ra, in.p[3] + off, t, lim);
  xrow_load<N, E, Cfg>(rb, in.p[4] + off, t, lim);
  xrow_inv<N, E, Cfg>(qx, ra, buf, t, tw, lim);
  GHX_PHASE();
  xrow_load<N, E, Cfg>(ra, in.p[5] + off, t, lim);
  xrow_inv<N, E, Cfg>(qy, rb, buf, t, tw, lim);
  GHX_PHASE();
  xrow_load<N, E, Cfg>(rb, in.p[0] + off, t, lim);
  xrow_inv<N, E, Cfg>(qz, ra, buf, t, tw, lim);
  GHX_PHASE();
  xrow_load<N, E, Cfg>(ra, in.p[1] + off, t, lim);
  {
    cplx px[E];
    xrow_inv<N, E, Cfg>(px, rb, buf, t, tw, lim);
#pragma unroll
    for (int m = 0; m < E; ++m) {
      ay[m] = c_make(qz[m].x * px[m].x, qz[m].y * px[m].y);  // Q_z P_x
      az[m] = c_make(px[m].x * qy[m].x, px[m].y * qy[m].y);  // P_x Q_y
    }
  }
  GHX_PHASE();
  xrow_load<N, E, Cfg>(rb, in.p[2] + off, t, lim);
  {
    cplx py[E];
    xrow_inv<N, E, Cfg>(py, ra, buf, t, tw, lim);
    cplx oz[E];
#pragma unroll
    for (int m = 0; m < E; ++m) {
      oz[m] = c_make((az[m].x - qx[m].x * py[m].x) * tmp, (az[m].y - qx[m].y * py[m].y) * tmp);
      az[m] = c_make(py[m].x * qz[m].x, py[m].y * qz[m].y);  // now P_y Q_z
    }
    xrow_fwd<N, E, Cfg>(oz, buf, t, tw, out.p[2] + off, lout);
  }
  GHX_PHASE();
  {
    cplx pz[E];
    xrow_inv<N, E, Cfg>(pz, rb, buf, t, tw, lim);
    cplx ox[E], oy[E];
#pragma unroll
    for (int m = 0; m < E; ++m) {
      ox[m] = c_make((az[m].x - qy[m].x * pz[m].x) * tmp, (az[m].y - qy[m].y * pz[m].y) * tmp);
      oy[m] = c_make((pz[m].x * qx[m].x - ay[m].x) * tmp, (pz[m].y * qx[m].y - ay[m].y) * tmp);
    }
    GHX_PHASE();
    xrow_fwd<N, E, Cfg>(ox, buf, t, tw, out.p[0] + off, lout);
    GHX_PHASE();
    xrow_fwd<N, E, Cfg>(oy, buf, t, tw, out.p[1] + off, lout);
  }
#undef GHX_PHASE
}

// Fused X^-1 . (A . B) tmp . X on P rows for advect3 (pseudospec3D_phd.f90:
// 23-115): in.p[0..2] = A, in.p[3..5] = B (grad of the scalar), out.p[0] =
// FFT[((A_x B_x + A_y B_y) + A_z B_z) tmp] with tmp = -1/N^6.
template <int N>
__global__ __launch_bounds__(kRowBound) void k_xdot(FieldSet in, FieldSet out, GridK g, int nxp,
                                             const cplx *__restrict__ twh, const cplx *__restrict__ twx, int kxin, int kxout, const unsigned *dirty) {
  const int kxlim = dirty && *dirty != 0u ? g.nxh : kxin;  // (as prune_input)
  using Cfg = FFTCfgLow<N>;
  constexpr int T = Cfg::T, E = Cfg::E;
  extern __shared__ cplx lds[];
  const int rpb = blockDim.x / T;
  const int lt = threadIdx.x / T, t = threadIdx.x % T;
  const long nrows = (long)g.nz * g.ny;
  const long r = (long)blockIdx.x * rpb + lt;
  const bool ok = r < nrows;
  if constexpr (T <= 64) {
    if (!ok) return;
  }
  const int lim = ok ? kxlim : 0, lout = ok ? kxout : 0;
  const size_t off = (size_t)(ok ? r : 0) * nxp;
  cplx *buf = lds + lt * lds_line_stride(N);
  const double tmp = -g.inv_n6;
  XTw<N, Cfg> tw;
  tw.load(twh, twx, t);
  XRowIn<E> ra, rb;
  cplx acc[E];
  xrow_load<N, E, Cfg>(ra, in.p[0] + off, t, lim);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    cplx a[E], b[E];
    xrow_load<N, E, Cfg>(rb, in.p[3 + d] + off, t, lim);
    xrow_inv<N, E, Cfg>(a, ra, buf, t, tw, lim);
    if (d < 2) xrow_load<N, E, Cfg>(ra, in.p[d + 1] + off, t, lim);
    xrow_inv<N, E, Cfg>(b, rb, buf, t, tw, lim);
#pragma unroll
    for (int m = 0; m < E; ++m) {
      const cplx p = c_make(a[m].x * b[m].x, a[m].y * b[m].y);
      if (d == 0) acc[m] = p;
      else if (d == 1) acc[m] = c_make(acc[m].x + p.x, acc[m].y + p.y);
      else acc[m] = c_make((acc[m].x + p.x) * tmp, (acc[m].y + p.y) * tmp);
    }
  }
  xrow_fwd<N, E, Cfg>(acc, buf, t, tw, out.p[0] + off, lout);
}

// ---------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------



#if GHX_PART == 2
// 512-point z lines on the 16-points-per-lane schedule: 8-line tiles (128-byte
// chunks of Q) from 256-lane blocks, for a pass that keeps one field live
template <int MODE>
static hipError_t launch_zinv_wide(const FFTCtx &c, int nf, const FieldSet &in, const FieldSet &out, int prune,
                                   const double *aux) {
  const GridK &g = c.gk;
  using Cfg = FFTCfgWide<512>;
  constexpr int T = Cfg::T;
  const PassShape s = wide_shape(T, lds_line_stride(512), g.ny);
  const int L = s.lines;
  dim3 grid((g.ny + L - 1) / L, g.nxh, c.batch);
  allow_lds(k_zinv<512, MODE, Cfg>, s.lds);
  GHX_LAUNCH_CHECK((k_zinv<512, MODE, Cfg>), s, kTileBound, T, true);
  hipLaunchKernelGGL((k_zinv<512, MODE, Cfg>), grid, dim3(L * T), s.lds, c.stream, in, out, nf, g, c.tw_z, prune_in(c, prune), prune_word(c, prune), aux);
  return hipGetLastError();
}

// the curl Z^-1 on the four-points-per-lane schedule (FFTCtx::sched bit 0)
template <int N>
static hipError_t launch_zinv_low(const FFTCtx &c, int nf, const FieldSet &in, const FieldSet &out, int prune,
                                  const double *aux) {
  const GridK &g = c.gk;
  using Cfg = FFTCfgLow<N>;
  constexpr int T = Cfg::T;
  const PassShape s = tile_shape(T, lds_line_stride(N), g.ny, tile_pick("GHX_LZ", c.tile_z, tile_default(T, 4)), max_lds());
  const int L = s.lines;
  dim3 grid((g.ny + L - 1) / L, g.nxh, c.batch);
  allow_lds(k_zinv<N, 1, Cfg>, s.lds);
  GHX_LAUNCH_CHECK((k_zinv<N, 1, Cfg>), s, kTileBound, T, true);
  hipLaunchKernelGGL((k_zinv<N, 1, Cfg>), grid, dim3(L * T), s.lds, c.stream, in, out, nf, g, c.tw_z, prune_in(c, prune), prune_word(c, prune), aux);
  return hipGetLastError();
}

static int zinv_outputs(int mode, int nf) {
  switch (mode) {
  case 1: case 4: return 6;
  case 2: return 12;
  case 5: case 6: return 9;
  case 7: return 3;
  default: return nf;
  }
}

hipError_t zinv(const FFTCtx &c, int mode, int nf, const FieldSet &in, const FieldSet &out, int prune,
                const double *aux) {
  if (mode == 3 && !aux) return hipErrorInvalidValue;
  const GridK &g = c.gk;
  if (mode == 0 || mode == 3 || mode == 7 ? z_lines(c) <= kSmallLines : small_z(c)) {
    const int nout = zinv_outputs(mode, nf);
    switch (g.nz) {
#define GHX_ONE(n_, Cfg_)                                                                    \
  {                                                                                         \
    constexpr int T = Cfg_::T;                                                              \
    const PassShape s = tile_shape(T, lds_line_stride(n_), g.ny, tile_pick("GHX_LZ", c.tile_z, tile_default(T, 4)), max_lds()); \
    allow_lds((k_zinv_one<n_, Cfg_>), s.lds);                                               \
    GHX_LAUNCH_CHECK((k_zinv_one<n_, Cfg_>), s, kTileBound, T, true);                       \
    hipLaunchKernelGGL((k_zinv_one<n_, Cfg_>), dim3((g.ny + s.lines - 1) / s.lines, g.nxh, c.batch * nout), dim3(s.block), s.lds, c.stream, in, out, mode, nout, g, c.tw_z, prune_in(c, prune), prune_word(c, prune), aux); \
    return hipGetLastError();                                                               \
  }
#define GHX_CASE(n_)                                                                        \
  case n_:                                                                                  \
    if constexpr (has_low<n_>()) if (mode == 1 && (c.sched & 1)) GHX_ONE(n_, FFTCfgLow<n_>) \
    GHX_ONE(n_, FFTCfgMix<n_>)
      GHX_SIZES(GHX_CASE)
#undef GHX_ONE
#undef GHX_CASE
    default: return hipErrorInvalidValue;
    }
  }
  if (mode == 1 && (c.sched & 1)) {
    switch (g.nz) {
    case 32: return launch_zinv_low<32>(c, nf, in, out, prune, aux);
    case 64: return launch_zinv_low<64>(c, nf, in, out, prune, aux);
    case 128: return launch_zinv_low<128>(c, nf, in, out, prune, aux);
    case 256: return launch_zinv_low<256>(c, nf, in, out, prune, aux);
    default: break;  // the same schedule either way
    }
  }
  // the spline prefilter pass at 512 points runs the wide schedule (GHX_ZWIDE=0
  // selects the default one); the plain and curl passes are slower on it
  if (mode == 3 && g.nz == 512 && env_switch("GHX_ZWIDE", 1) != 0 &&
      wide_shape(FFTCfgWide<512>::T, lds_line_stride(512), g.ny).lds <= max_lds())
    return launch_zinv_wide<3>(c, nf, in, out, prune, aux);
  if (mode == 0 || mode == 3) {
    switch (g.nz) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    using Cfg = ZInvCfg<n_>;                                                                \
    constexpr int T = Cfg::T;                                                               \
    const PassShape s = tile_shape(T, lds_line_stride(n_), g.ny, tile_pick("GHX_LZ", c.tile_z, tile_default(T, 8)), max_lds()); \
    const dim3 grid((g.ny + s.lines - 1) / s.lines, g.nxh, c.batch);                        \
    if (mode == 0) {                                                                        \
      allow_lds((k_zinv<n_, 0, Cfg>), s.lds);                                               \
      GHX_LAUNCH_CHECK((k_zinv<n_, 0, Cfg>), s, kTileBound, T, true);                       \
      hipLaunchKernelGGL((k_zinv<n_, 0, Cfg>), grid, dim3(s.block), s.lds, c.stream, in, out, nf, g, c.tw_z, prune_in(c, prune), prune_word(c, prune), aux); \
    } else {                                                                                \
      allow_lds((k_zinv<n_, 3, Cfg>), s.lds);                                               \
      GHX_LAUNCH_CHECK((k_zinv<n_, 3, Cfg>), s, kTileBound, T, true);                       \
      hipLaunchKernelGGL((k_zinv<n_, 3, Cfg>), grid, dim3(s.block), s.lds, c.stream, in, out, nf, g, c.tw_z, prune_in(c, prune), prune_word(c, prune), aux); \
    }                                                                                       \
    return hipGetLastError();                                                               \
  }
      GHX_SIZES(GHX_CASE)
#undef GHX_CASE
    default: return hipErrorInvalidValue;
    }
  }
  // Several fields: 8 lines (128-byte chunks of Q) while that is at most 256
  // lanes, else 4; the curl alone 8.  4 against 8 lines, us: curl 95.7 | 81.6 at
  // 256^3, 282 | 236 at 512 x 512 x 192, 166 | 137 at 384 x 384 x 192, MHD 299 | 256 at
  // 256 x 384 x 256, Boussinesq 127 | 107 at 384 x 384 x 96 (but 22.6 | 24.1 for the
  // curl at 128 x 128 x 192, 40.3 | 42.2 at 192^3); of 64 lanes HD 394 | 438 at 384^3,
  // MHD 633 | 648 at 256 x 256 x 512; the curl alone 225 | 181 at 256^3.
  switch (g.nz) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    constexpr int T = FFTCfg<n_>::T;                                                        \
    const PassShape s = tile_shape(T, lds_line_stride(n_), g.ny, tile_pick("GHX_LZ", c.tile_z, tile_default(T, mode == 7 || T <= 32 ? 8 : 4)), max_lds()); \
    const int L = s.lines; const size_t lds = s.lds;                            \
    dim3 grid((g.ny + L - 1) / L, g.nxh, c.batch);                                          \
    if (mode == 1) {                                                                 \
      allow_lds(k_zinv<n_, 1>, lds);                                                        \
      GHX_LAUNCH_CHECK((k_zinv<n_, 1>), s, kTileBound, T, true); hipLaunchKernelGGL((k_zinv<n_, 1>), grid, dim3(L * T), lds, c.stream, in, out, nf, g, c.tw_z, prune_in(c, prune), prune_word(c, prune), aux); \
    } else if (mode == 2) {                                                                 \
      allow_lds(k_zinv<n_, 2>, lds);                                                        \
      GHX_LAUNCH_CHECK((k_zinv<n_, 2>), s, kTileBound, T, true); hipLaunchKernelGGL((k_zinv<n_, 2>), grid, dim3(L * T), lds, c.stream, in, out, nf, g, c.tw_z, prune_in(c, prune), prune_word(c, prune), aux); \
    } else if (mode == 4) {                                                                 \
      allow_lds(k_zinv<n_, 4>, lds);                                                        \
      GHX_LAUNCH_CHECK((k_zinv<n_, 4>), s, kTileBound, T, true); hipLaunchKernelGGL((k_zinv<n_, 4>), grid, dim3(L * T), lds, c.stream, in, out, nf, g, c.tw_z, prune_in(c, prune), prune_word(c, prune), aux); \
    } else if (mode == 5) {                                                                 \
      allow_lds(k_zinv<n_, 5>, lds);                                                        \
      GHX_LAUNCH_CHECK((k_zinv<n_, 5>), s, kTileBound, T, true); hipLaunchKernelGGL((k_zinv<n_, 5>), grid, dim3(L * T), lds, c.stream, in, out, nf, g, c.tw_z, prune_in(c, prune), prune_word(c, prune), aux); \
    } else if (mode == 6) {                                                                 \
      allow_lds(k_zinv<n_, 6>, lds);                                                        \
      GHX_LAUNCH_CHECK((k_zinv<n_, 6>), s, kTileBound, T, true); hipLaunchKernelGGL((k_zinv<n_, 6>), grid, dim3(L * T), lds, c.stream, in, out, nf, g, c.tw_z, prune_in(c, prune), prune_word(c, prune), aux); \
    } else if (mode == 7) {                                                                 \
      allow_lds(k_zinv<n_, 7>, lds);                                                        \
      GHX_LAUNCH_CHECK((k_zinv<n_, 7>), s, kTileBound, T, true); hipLaunchKernelGGL((k_zinv<n_, 7>), grid, dim3(L * T), lds, c.stream, in, out, nf, g, c.tw_z, prune_in(c, prune), prune_word(c, prune), aux); \
    }                                                                                       \
    break;                                                                                  \
  }
    GHX_SIZES(GHX_CASE)
#undef GHX_CASE
  default:
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

#endif

#if GHX_PART == 3
hipError_t zfwd(const FFTCtx &c, int nf, const FieldSet &in, const FieldSet &out, int prune) {
  const GridK &g = c.gk;
  switch (g.nz) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    using Cfg = FFTCfgMix<n_>;                                                              \
    constexpr int T = Cfg::T;                                                               \
    const PassShape s = tile_shape(T, lds_line_stride(n_), g.ny, tile_want("GHX_LZ", tile_default(T, 8)), max_lds());                                        \
    const int L = s.lines; const size_t lds = s.lds;                            \
    dim3 grid((g.ny + L - 1) / L, g.nxh);                                                   \
    allow_lds((k_zfwd<n_, Cfg>), lds);                                                             \
    GHX_LAUNCH_CHECK((k_zfwd<n_, Cfg>), s, kTileBound, T, true); hipLaunchKernelGGL((k_zfwd<n_, Cfg>), grid, dim3(L * T), lds, c.stream, in, out, nf, g, c.tw_z, prune); \
    break;                                                                                  \
  }
    GHX_SIZES(GHX_CASE)
#undef GHX_CASE
  default:
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

#endif

template <int N, int KIND, typename Cfg>
static hipError_t launch_zrk(const FFTCtx &c, const FieldSet &in, const ZUpdate &u, int prune, int nz) {
  constexpr int T = Cfg::T, G = zrk_groups(KIND);
  const GridK &g = c.gk;
  // up to 4 lines; the Boussinesq block at most 256 lanes (212 -> 177 us at
  // 256^3 with 2 lines instead of 4)
  const int want = KIND == 2 && G * T * 4 > 256 ? 2 : 4;
  const PassShape s = zrk_shape(G, T, zrk_bound(KIND), lds_line_stride(N), g.ny, tile_pick("GHX_LZ", c.tile_z, want), max_lds());
  const int L = s.lines;
  allow_lds(k_zrk<N, KIND, Cfg>, s.lds);
  GHX_LAUNCH_CHECK((k_zrk<N, KIND, Cfg>), s, zrk_bound(KIND), T, true);
  hipLaunchKernelGGL((k_zrk<N, KIND, Cfg>), dim3((g.ny + L - 1) / L, g.nxh, nz), dim3(s.block), s.lds, c.stream, in, g,
                     c.tw_z, u, prune);
  return hipGetLastError();
}

#if GHX_PART == 4
hipError_t zfwd_rk_hd(const FFTCtx &c, const FieldSet &in, const RKParams &rk, int prune) {
  const GridK &g = c.gk;
  // 512-point lines take the four-points-per-lane schedule by default (128
  // lanes per line, four lines per 512-lane block): 124 registers per lane
  // against 224, two blocks per CU, so the update's loads of v and C overlap
  // more (0.71 -> 0.70 ms at 512^3; GHX_ZLOW=0 selects the default schedule).
  // Other sizes take it on request (FFTCtx::sched bit 0).
  const bool low = (c.sched & 1) || (g.nz == 512 && env_switch("GHX_ZLOW", 1) == 1);
  if (small_z(c) && takes_zrk(zrk_groups(0), lds_line_stride(g.nz), max_lds())) {
    ZUpdate u{};
    u.dt = rk.dt; u.rmp = rk.rmp; u.om2 = rk.om2; u.nu = rk.nu;
    u.fline = rk.fline; u.bstride = rk.bstride; u.nu_b = rk.nu_b;
    for (int k = 0; k < 3; ++k) { u.v[k] = rk.v[k]; u.c[k] = rk.c[k]; u.f[k] = rk.f[k]; u.out[k] = rk.out[k]; }
    switch (g.nz) {
#define GHX_CASE(n_)                                                                        \
  case n_:                                                                                  \
    if constexpr (has_low<n_>()) if (low) return launch_zrk<n_, 0, FFTCfgLow<n_>>(c, in, u, prune, c.batch); \
    return launch_zrk<n_, 0, FFTCfgMix<n_>>(c, in, u, prune, c.batch);
      GHX_SIZES(GHX_CASE)
#undef GHX_CASE
    default: return hipErrorInvalidValue;
    }
  }
  // On the four-points-per-lane schedule the next field's Q tile is loaded
  // while this one is transformed (138 registers against 124; 0.698 -> 0.671
  // ms at 512^3; GHX_ZPF=0 loads one tile at a time)
  const int pf = env_switch("GHX_ZPF", 1) != 0 ? 1 : 0;
  if (low) {
    switch (g.nz) {
#define GHX_LOW(n_)                                                                                     \
  case n_: {                                                                                            \
    using Cfg = FFTCfgLow<n_>;                                                                          \
    constexpr int T = Cfg::T;                                                                           \
    const PassShape s = tile_shape(T, lds_line_stride(n_), g.ny, tile_pick("GHX_LZ", c.tile_z, tile_default(T, 4)), max_lds()); \
    const int L = s.lines;                                                                              \
    dim3 grid((g.ny + L - 1) / L, g.nxh, c.batch);                                                      \
    if (pf) {                                                                                           \
      allow_lds(k_zfwd_rk_hd<n_, Cfg, 1>, s.lds);                                                       \
      GHX_LAUNCH_CHECK((k_zfwd_rk_hd<n_, Cfg, 1>), s, kTileBound, T, true);                             \
      hipLaunchKernelGGL((k_zfwd_rk_hd<n_, Cfg, 1>), grid, dim3(L * T), s.lds, c.stream, in, g, c.tw_z, rk, prune); \
    } else {                                                                                            \
      allow_lds(k_zfwd_rk_hd<n_, Cfg>, s.lds);                                                          \
      GHX_LAUNCH_CHECK((k_zfwd_rk_hd<n_, Cfg>), s, kTileBound, T, true);                                \
      hipLaunchKernelGGL((k_zfwd_rk_hd<n_, Cfg>), grid, dim3(L * T), s.lds, c.stream, in, g, c.tw_z, rk, prune); \
    }                                                                                                   \
    return hipGetLastError();                                                                           \
  }
      GHX_LOW(32) GHX_LOW(64) GHX_LOW(128) GHX_LOW(256) GHX_LOW(512)
#undef GHX_LOW
    default:
      break;  // the same schedule either way
    }
  }
  switch (g.nz) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    constexpr int T = FFTCfg<n_>::T;                                                        \
    const PassShape s = tile_shape(T, lds_line_stride(n_), g.ny, tile_pick("GHX_LZ", c.tile_z, tile_default(T, 4)), max_lds());         \
    const int L = s.lines; const size_t lds = s.lds;                            \
    dim3 grid((g.ny + L - 1) / L, g.nxh, c.batch);                                          \
    allow_lds(k_zfwd_rk_hd<n_>, lds);                                                       \
    GHX_LAUNCH_CHECK((k_zfwd_rk_hd<n_>), s, kTileBound, T, true); hipLaunchKernelGGL((k_zfwd_rk_hd<n_>), grid, dim3(L * T), lds, c.stream, in, g, c.tw_z, rk, prune); \
    break;                                                                                  \
  }
    GHX_SIZES(GHX_CASE)
#undef GHX_CASE
  default:
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

#endif

#if GHX_PART == 5
hipError_t zfwd_rk_mhd(const FFTCtx &c, const FieldSet &in, const MHDRKParams &rk, int prune) {
  const GridK &g = c.gk;
  const bool low = env_switch("GHX_ZLOW", 1) == 1;
  if (small_z(c) && takes_zrk(zrk_groups(1), lds_line_stride(g.nz), max_lds())) {
    ZUpdate u{};
    u.dt = rk.dt; u.rmp = rk.rmp; u.nu = rk.nu; u.mu = rk.mu; u.fline = rk.fline;
    for (int k = 0; k < 6; ++k) { u.v[k] = rk.v[k]; u.c[k] = rk.c[k]; u.f[k] = rk.f[k]; u.out[k] = rk.out[k]; }
    switch (g.nz) {
#define GHX_CASE(n_)                                                                        \
  case n_:                                                                                  \
    if constexpr (has_low<n_>()) if (low) return launch_zrk<n_, 1, FFTCfgLow<n_>>(c, in, u, prune, 2); \
    return launch_zrk<n_, 1, FFTCfgMix<n_>>(c, in, u, prune, 2);
      GHX_SIZES(GHX_CASE)
#undef GHX_CASE
    default: return hipErrorInvalidValue;
    }
  }
  // the four-points-per-lane schedule where a size has one (GHX_ZLOW=0: the
  // default schedule); 8 lines to 256 lanes, else 4 (both parts together, 4 | 8
  // lines: 103 | 87 us at 384 x 384 x 48, 53 | 52 at 256 x 256 x 48, from 96 points on
  // within 5% either way; of 64 lanes 764 | 814 at 512 x 512 x 256)
  switch (g.nz) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    if constexpr (FFTCfgLow<n_>::E != FFTCfg<n_>::E) if (low) {                              \
      using Cl = FFTCfgLow<n_>;                                                              \
      constexpr int T = Cl::T;                                                               \
      const PassShape s = tile_shape(T, lds_line_stride(n_), g.ny, tile_want("GHX_LZ", tile_default(T, T <= 32 ? 8 : 4)), max_lds()); \
      const int L = s.lines; const size_t lds = s.lds;                                       \
      dim3 grid((g.ny + L - 1) / L, g.nxh);                                                  \
      allow_lds(k_zfwd_rk_mhd<n_, 0, Cl>, lds);                                              \
      allow_lds(k_zfwd_rk_mhd<n_, 1, Cl>, lds);                                              \
      GHX_LAUNCH_CHECK((k_zfwd_rk_mhd<n_, 0, Cl>), s, kTileBound, T, true);                  \
      hipLaunchKernelGGL((k_zfwd_rk_mhd<n_, 0, Cl>), grid, dim3(L * T), lds, c.stream, in, g, c.tw_z, rk, prune); \
      GHX_LAUNCH_CHECK((k_zfwd_rk_mhd<n_, 1, Cl>), s, kTileBound, T, true);                  \
      hipLaunchKernelGGL((k_zfwd_rk_mhd<n_, 1, Cl>), grid, dim3(L * T), lds, c.stream, in, g, c.tw_z, rk, prune); \
      break;                                                                                 \
    }                                                                                        \
    constexpr int T = FFTCfg<n_>::T;                                                        \
    const PassShape s = tile_shape(T, lds_line_stride(n_), g.ny, tile_want("GHX_LZ", tile_default(T, T <= 32 ? 8 : 4)), max_lds());                                        \
    const int L = s.lines; const size_t lds = s.lds;                            \
    dim3 grid((g.ny + L - 1) / L, g.nxh);                                                   \
    allow_lds(k_zfwd_rk_mhd<n_, 0>, lds);                                                   \
    allow_lds(k_zfwd_rk_mhd<n_, 1>, lds);                                                   \
    GHX_LAUNCH_CHECK((k_zfwd_rk_mhd<n_, 0>), s, kTileBound, T, true); hipLaunchKernelGGL((k_zfwd_rk_mhd<n_, 0>), grid, dim3(L * T), lds, c.stream, in, g, c.tw_z, rk, prune); \
    GHX_LAUNCH_CHECK((k_zfwd_rk_mhd<n_, 1>), s, kTileBound, T, true); hipLaunchKernelGGL((k_zfwd_rk_mhd<n_, 1>), grid, dim3(L * T), lds, c.stream, in, g, c.tw_z, rk, prune); \
    break;                                                                                  \
  }
    GHX_SIZES(GHX_CASE)
#undef GHX_CASE
  default:
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

#endif

#if GHX_PART == 1
// the y passes on the four-points-per-lane schedule (FFTCtx::sched bit 1)
template <int N>
static hipError_t launch_y_low(const FFTCtx &c, bool inv, int nf, const FieldSet &in, const FieldSet &out, int prune) {
  const GridK &g = c.gk;
  const YSplit sp = ysplit(small_y(c), nf, c.batch);
  using Cfg = FFTCfgLow<N>;
  constexpr int T = Cfg::T;
  const int nxp = p_row(g);
  const PassShape s = tile_shape(T, lds_line_stride(N), g.nxh, tile_pick("GHX_LY", c.tile_y, tile_default(T, inv ? 8 : 4)), max_lds());
  const int L = s.lines;
  dim3 grid((g.nxh + L - 1) / L, g.nz, c.batch * sp.parts);
  if (inv) {
    allow_lds(k_yinv<N, Cfg>, s.lds);
    GHX_LAUNCH_CHECK((k_yinv<N, Cfg>), s, kTileBound, T, true);
    hipLaunchKernelGGL((k_yinv<N, Cfg>), grid, dim3(L * T), s.lds, c.stream, in, out, nf, sp, g, nxp, c.tw_y, kx_in(c, prune), prune_in(c, prune), prune_word(c, prune));
  } else {
    allow_lds(k_yfwd<N, Cfg>, s.lds);
    GHX_LAUNCH_CHECK((k_yfwd<N, Cfg>), s, kTileBound, T, true);
    hipLaunchKernelGGL((k_yfwd<N, Cfg>), grid, dim3(L * T), s.lds, c.stream, in, out, nf, sp, g, nxp, c.tw_y, kx_out(c, prune), prune);
  }
  return hipGetLastError();
}
static bool y_low(const FFTCtx &c, bool inv, int nf, const FieldSet &in, const FieldSet &out, int prune,
                  hipError_t *err) {
  if (!(c.sched & 2)) return false;
  switch (c.gk.ny) {
  case 32: *err = launch_y_low<32>(c, inv, nf, in, out, prune); return true;
  case 64: *err = launch_y_low<64>(c, inv, nf, in, out, prune); return true;
  case 128: *err = launch_y_low<128>(c, inv, nf, in, out, prune); return true;
  case 256: *err = launch_y_low<256>(c, inv, nf, in, out, prune); return true;
  default: return false;  // the same schedule either way, or the wide 512-point pass
  }
}

hipError_t yinv(const FFTCtx &c, int nf, const FieldSet &in, const FieldSet &out, int prune) {
  const GridK &g = c.gk;
  const long lines = (long)g.kxact * g.nz * c.batch;
  const YSplit sp = ysplit(small_y(c) || long_y(g.ny, nf, lines, prune != 0), nf, c.batch);
  const int nxp = p_row(g);
  hipError_t lerr;
  if (y_low(c, true, nf, in, out, prune, &lerr)) return lerr;
  switch (g.ny) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    using Cfg = YInvCfg<n_>;                                                                \
    constexpr int T = Cfg::T;                                                               \
    if constexpr (FFTCfgWide<n_>::E != FFTCfg<n_>::E)                                        \
    if (env_switch("GHX_YWIDE", 1) == 1 &&                                                   \
        wide_shape(FFTCfgWide<n_>::T, lds_line_stride(n_), g.nxh).lds <= max_lds()) {         \
      /* 16 points per lane: 8-line tiles from 256-lane blocks, two blocks per CU */       \
      constexpr int TW = FFTCfgWide<n_>::T;                                                  \
      const PassShape s = wide_shape(TW, lds_line_stride(n_), g.nxh);                        \
      const int L = s.lines; const size_t lds = s.lds;                                       \
      dim3 grid((g.nxh + L - 1) / L, g.nz, c.batch * sp.parts);                                         \
      GHX_LAUNCH_CHECK((k_yinv<n_, FFTCfgWide<n_>>), s, kTileBound, TW, true);               \
      allow_lds(k_yinv<n_, FFTCfgWide<n_>>, lds);                                            \
      hipLaunchKernelGGL((k_yinv<n_, FFTCfgWide<n_>>), grid, dim3(L * TW), lds, c.stream, in, out, nf, sp, g, nxp, \
                         c.tw_y, kx_in(c, prune), prune_in(c, prune), prune_word(c, prune));                                              \
      break;                                                                                 \
    }                                                                                        \
    const PassShape s = tile_shape(T, lds_line_stride(n_), g.nxh, tile_pick("GHX_LY", c.tile_y, tile_default(T, 8)), max_lds());        \
    const int L = s.lines; const size_t lds = s.lds;                            \
    dim3 grid((g.nxh + L - 1) / L, g.nz, c.batch * sp.parts);                                          \
    allow_lds(k_yinv<n_, Cfg>, lds);                                                             \
    GHX_LAUNCH_CHECK((k_yinv<n_, Cfg>), s, kTileBound, T, true); hipLaunchKernelGGL((k_yinv<n_, Cfg>), grid, dim3(L * T), lds, c.stream, in, out, nf, sp, g, nxp, c.tw_y, kx_in(c, prune), prune_in(c, prune), prune_word(c, prune)); \
    break;                                                                                  \
  }
    GHX_SIZES(GHX_CASE)
#undef GHX_CASE
  default:
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t yfwd(const FFTCtx &c, int nf, const FieldSet &in, const FieldSet &out, int prune) {
  const GridK &g = c.gk;
  const YSplit sp = ysplit(small_y(c), nf, c.batch);
  const int nxp = p_row(g);
  hipError_t lerr;
  if (y_low(c, false, nf, in, out, prune, &lerr)) return lerr;
  switch (g.ny) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    using Cfg = YFwdCfg<n_>;                                                                \
    constexpr int T = Cfg::T;                                                               \
    const PassShape s = tile_shape(T, lds_line_stride(n_), g.nxh, tile_pick("GHX_LY", c.tile_y, tile_default(T, Cfg::E == 12 ? 8 : 4)), max_lds());        \
    const int L = s.lines; const size_t lds = s.lds;                            \
    dim3 grid((g.nxh + L - 1) / L, g.nz, c.batch * sp.parts);                                          \
    allow_lds(k_yfwd<n_, Cfg>, lds);                                                             \
    GHX_LAUNCH_CHECK((k_yfwd<n_, Cfg>), s, kTileBound, T, true); hipLaunchKernelGGL((k_yfwd<n_, Cfg>), grid, dim3(L * T), lds, c.stream, in, out, nf, sp, g, nxp, c.tw_y, kx_out(c, prune), prune); \
    break;                                                                                  \
  }
    GHX_SIZES(GHX_CASE)
#undef GHX_CASE
  default:
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
#endif

#if GHX_PART == 6

hipError_t xinv(const FFTCtx &c, int nf, const FieldSet &in, double *const *out, int prune) {
  const GridK &g = c.gk;
  if (g.nx % 2) return hipErrorInvalidValue;
  const int kxlim = prune == 1 ? g.kxact : g.nxh;
  RealSet rs;
  for (int f = 0; f < nf; ++f) rs.p[f] = out[f];
  const long nrows = (long)g.nz * g.ny;
  const int nxp = p_row(g);
  if (use_x2(g.nx)) {
    switch (g.nx) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    constexpr int T = FFTCfg<n_>::T;                                                        \
    const PassShape s = row_shape(T, lds_line_stride(n_), max_lds(), nrows);                                        \
    const int rpb = s.lines; const size_t lds = s.lds;                                      \
    const dim3 bl(rpb * T);                                                                 \
    if (nf > 1) { /* pairs of fields, the last of an odd count alone */                     \
      GHX_LAUNCH_CHECK((k_xinv2<n_>), s, kRowBound, T, false);                              \
      hipLaunchKernelGGL((k_xinv2<n_>), dim3((unsigned)((nrows + rpb - 1) / rpb)), bl, lds, c.stream, in, rs, nf, g, nxp, c.tw_x, kxlim); \
    } else { /* a lone field's rows in pairs */                                             \
      GHX_LAUNCH_CHECK((k_xinv_rows<n_>), s, kRowBound, T, false);                          \
      hipLaunchKernelGGL((k_xinv_rows<n_>), dim3((unsigned)((nrows + 2 * rpb - 1) / (2 * rpb))), bl, lds, c.stream, in.p[0], rs.p[0], nrows, nxp, c.tw_x, kxlim); \
    }                                                                                       \
    return hipGetLastError();                                                               \
  }
      GHX_X2_SIZES(GHX_CASE)
#undef GHX_CASE
      default:
        break;
    }
  }
  switch (g.nx / 2) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    constexpr int T = FFTCfgLow<n_>::T;                                                     \
    const PassShape s = row_shape(T, lds_line_stride(n_), max_lds(), nrows);                                        \
    const int rpb = s.lines; const size_t lds = s.lds;                          \
    GHX_LAUNCH_CHECK((k_xinv<n_>), s, kRowBound, T, false); hipLaunchKernelGGL((k_xinv<n_>), dim3((unsigned)((nrows + rpb - 1) / rpb)), dim3(rpb * T), lds, c.stream, in, rs, nf, g, nxp, c.tw_xh, c.tw_x, kxlim); \
    break;                                                                                  \
  }
    GHX_SIZES(GHX_CASE)
#undef GHX_CASE
  default:
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t xinv3i(const FFTCtx &c, const FieldSet &in, double *out, int prune) {
  const GridK &g = c.gk;
  if (g.nx % 2) return hipErrorInvalidValue;
  const int kxlim = prune == 1 ? g.kxact : g.nxh;
  const long nrows = (long)g.nz * g.ny;
  const int nxp = p_row(g);
  if (use_x2(g.nx)) {
    switch (g.nx) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    constexpr int T = FFTCfg<n_>::T;                                                        \
    const PassShape s = row_shape(T, lds_line_stride(n_), max_lds(), nrows);                                        \
    const int rpb = s.lines; const size_t lds = s.lds;                          \
    const dim3 gr((unsigned)((nrows + rpb - 1) / rpb)), bl(rpb * T);                      \
    GHX_LAUNCH_CHECK((k_xinv3i2<n_>), s, kRowBound, T, false); hipLaunchKernelGGL((k_xinv3i2<n_>), gr, bl, lds, c.stream, in, out, g, nxp, c.tw_x, kxlim);                                                                 \
    return hipGetLastError();                                                               \
  }
      GHX_X2_SIZES(GHX_CASE)
#undef GHX_CASE
      default:
        break;
    }
  }
  switch (g.nx / 2) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    constexpr int T = FFTCfgLow<n_>::T;                                                     \
    const PassShape s = row_shape(T, lds_line_stride(n_), max_lds(), nrows);                                        \
    const int rpb = s.lines; const size_t lds = s.lds;                          \
    GHX_LAUNCH_CHECK((k_xinv3i<n_>), s, kRowBound, T, false); hipLaunchKernelGGL((k_xinv3i<n_>), dim3((unsigned)((nrows + rpb - 1) / rpb)), dim3(rpb * T), lds, c.stream, in, out, g, nxp, c.tw_xh, c.tw_x, kxlim); \
    break;                                                                                  \
  }
    GHX_SIZES(GHX_CASE)
#undef GHX_CASE
  default:
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t xnormmax(const FFTCtx &c, const FieldSet &in, double *part, int *nblk) {
  const GridK &g = c.gk;
  if (g.nx % 2) return hipErrorInvalidValue;
  if (!use_x2(g.nx)) return hipErrorNotSupported;
  const long nrows = (long)g.nz * g.ny;
  switch (g.nx) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    constexpr int T = FFTCfg<n_>::T;                                                        \
    const PassShape s = row_shape(T, lds_line_stride(n_), max_lds() - kRowBound * sizeof(double)); \
    const long nb = (nrows + s.lines - 1) / s.lines;                                        \
    *nblk = (int)(nb < kNormBlocks ? nb : kNormBlocks);                                     \
    GHX_LAUNCH_CHECK((k_xnorm2<n_>), s, kRowBound, T, false);                               \
    hipLaunchKernelGGL((k_xnorm2<n_>), dim3(*nblk), dim3(s.block), s.lds, c.stream, in, part, g, p_row(g), c.tw_x, g.nxh); \
    return hipGetLastError();                                                               \
  }
    GHX_X2_SIZES(GHX_CASE)
#undef GHX_CASE
  default:
    return hipErrorNotSupported;
  }
}

hipError_t xfwd(const FFTCtx &c, int nf, const double *const *in, const FieldSet &out) {
  const GridK &g = c.gk;
  if (g.nx % 2) return hipErrorInvalidValue;
  RealSet rs;
  for (int f = 0; f < nf; ++f) rs.p[f] = const_cast<double *>(in[f]);
  const long nrows = (long)g.nz * g.ny;
  const int nxp = p_row(g);
  if (use_x2(g.nx)) {
    switch (g.nx) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    constexpr int T = FFTCfg<n_>::T;                                                        \
    const PassShape s = row_shape(T, lds_line_stride(n_), max_lds(), nrows);                                        \
    const int rpb = s.lines; const size_t lds = s.lds;                                      \
    const dim3 bl(rpb * T);                                                                 \
    bool paired = false;                                                                    \
    if constexpr (pair_rows_fwd(n_)) paired = nf == 1;                                      \
    if (paired) {                                                                           \
      GHX_LAUNCH_CHECK((k_xfwd_rows<n_>), s, kRowBound, T, false);                          \
      hipLaunchKernelGGL((k_xfwd_rows<n_>), dim3((unsigned)((nrows + 2 * rpb - 1) / (2 * rpb))), bl, lds, c.stream, rs.p[0], out.p[0], nrows, nxp, c.tw_x); \
    } else {                                                                                \
      GHX_LAUNCH_CHECK((k_xfwd2<n_>), s, kRowBound, T, false);                              \
      hipLaunchKernelGGL((k_xfwd2<n_>), dim3((unsigned)((nrows + rpb - 1) / rpb)), bl, lds, c.stream, rs, out, nf, g, nxp, c.tw_x); \
    }                                                                                       \
    return hipGetLastError();                                                               \
  }
      GHX_X2_SIZES(GHX_CASE)
#undef GHX_CASE
      default:
        break;
    }
  }
  switch (g.nx / 2) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    constexpr int T = FFTCfgLow<n_>::T;                                                     \
    const PassShape s = row_shape(T, lds_line_stride(n_), max_lds(), nrows);                                        \
    const int rpb = s.lines; const size_t lds = s.lds;                          \
    GHX_LAUNCH_CHECK((k_xfwd<n_>), s, kRowBound, T, false); hipLaunchKernelGGL((k_xfwd<n_>), dim3((unsigned)((nrows + rpb - 1) / rpb)), dim3(rpb * T), lds, c.stream, rs, out, nf, g, nxp, c.tw_xh, c.tw_x); \
    break;                                                                                  \
  }
    GHX_SIZES(GHX_CASE)
#undef GHX_CASE
  default:
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
#endif

#if GHX_PART == 9
// ---------------------------------------------------------------------------
// Small planes: X and Y of one field's (x, y) plane in one block, the plane held
// in LDS between them (one line of y per kx), so the P array is neither written
// nor read and a launch of three goes.  Rows go in pairs of the field's own (NY
// is even).  Sides of 24 to 64 points: at most 76 KB of LDS, two blocks per CU;
// 96 x 96 points would leave one.  Whole transforms, separate passes -> planes,
// r2c and c2r, us: 13.2 -> 9.1 and 9.9 -> 9.2 at 32^3, 13.0 -> 10.8 and 11.9 ->
// 10.5 at 64^3, 23.2 -> 16.0 and 21.7 -> 14.9 at 64 x 64 x 256; of several
// fields 22.5 -> 14.7 and 15.7 -> 9.5 (6 of 32^3), 72.9 -> 52.2 and 63.7 -> 42.9
// (3 of 64 x 64 x 512).  prune (inverse): as in k_yinv, q holds data on the
// dealias set's lines only; the forward writes every line.  Rows at their own
// scale as in k_xinv_rows, and every twiddle power read: c2r 10.3 -> 10.6 us,
// r2c 9.95 -> 9.8 at 64^3, errors 4.29 -> 3.41e-16 and 4.36 -> 3.40e-16.
// ---------------------------------------------------------------------------
template <int NX, int NY, bool FWD>
__global__ __launch_bounds__(kRowBound) void k_xyplane(RealSet re, FieldSet q, GridK g, const cplx *__restrict__ twx,
                                                       const cplx *__restrict__ twy, int prune) {
  using X = Line<NX, FFTCfgRoots<FFTCfgMix<NX>, true>>;
  using Y = Line<NY, FFTCfgRoots<FFTCfgMix<NY>, true>>;
  static_assert(X::T <= 64 && Y::T <= 64 && NY % 2 == 0, "lines within a wavefront, rows in pairs");
  constexpr int H = NX / 2 + 1, SX = lds_line_stride(NX), SY = lds_line_stride(NY);
  constexpr int LX = (int)kRowBound / X::T, LY = (int)kRowBound / Y::T;
  extern __shared__ cplx lds[];
  cplx *plane = lds + LX * SX;  // H lines of SY points
  const int z = blockIdx.x;
  double *real = re.p[blockIdx.y] + (size_t)z * NY * NX;
  cplx *spec = q.p[blockIdx.y] + (size_t)z * H * NY;
  auto rows = [&]() {
    const int t = threadIdx.x % X::T;
    cplx *buf = lds + (threadIdx.x / X::T) * SX;
    X fft;
    if constexpr (FWD) fft.load_fwd(twx, t);
    else fft.load_inv(twx, t);
    for (int p = threadIdx.x / X::T; p < NY / 2; p += LX) {
      double *r0 = real + (size_t)(2 * p) * NX, *r1 = r0 + NX;
      cplx x[X::SE], k[X::KE];
      if constexpr (FWD) {
        if (X::live(t)) xpair_real<X::SE>(x, r0, r1, t, X::A);
        fft.fwd(x, k, buf, t);
#pragma unroll
        for (int m = 0; m < X::KE; ++m) buf[lds_pad(t + X::T * m)] = k[m];
        line_sync<X::T>();
#pragma unroll
        for (int m = 0; m <= X::KE / 2; ++m) {
          const int i = t + X::T * m;
          if (i < H) {
            const cplx c = c_conj(buf[lds_pad((NX - i) % NX)]);
            const cplx d = c_sub(k[m], c);
            plane[i * SY + lds_pad(2 * p)] = c_scale(c_add(k[m], c), 0.5);
            plane[i * SY + lds_pad(2 * p + 1)] = c_make(0.5 * d.y, -0.5 * d.x);
          }
        }
        line_sync<X::T>();
      } else {
        cplx a[X::KE], b[X::KE];
#pragma unroll
        for (int m = 0; m < X::KE; ++m) {
          const int i = t + X::T * m, c = i < H ? i : NX - i;
          a[m] = plane[c * SY + lds_pad(2 * p)];
          b[m] = plane[c * SY + lds_pad(2 * p + 1)];
        }
        RowScale ra, rb;
        xpair_make_scaled<NX, X::KE, X::T>(k, a, b, t, H, true, ra, rb);
        fft.inv(k, x, buf, t);
        if (X::live(t)) {
#pragma unroll
          for (int m = 0; m < X::SE; ++m) {
            r0[t + X::A * m] = x[m].x * ra.out;
            r1[t + X::A * m] = x[m].y * rb.out;
          }
        }
      }
    }
  };
  auto lines = [&]() {
    const int t = threadIdx.x % Y::T;
    Y fft;
    if constexpr (FWD) fft.load_fwd(twy, t);
    else fft.load_inv(twy, t);
    for (int i = threadIdx.x / Y::T; i < H; i += LY) {
      cplx *row = plane + i * SY, *s = spec + (size_t)i * NY;
      cplx x[Y::SE], k[Y::KE];
      if constexpr (FWD) {
        Y::get(x, row, t);
        line_sync<Y::T>();
        fft.fwd(x, k, row, t);
#pragma unroll
        for (int m = 0; m < Y::KE; ++m) s[t + Y::T * m] = k[m];
      } else {
#pragma unroll
        for (int m = 0; m < Y::KE; ++m) {
          const int j = t + Y::T * m;
          const bool need = !prune || kn2_of(g, i, j, 0) <= g.kmax;
          const cplx v = s[need ? j : 0];
          k[m] = need ? v : c_make(0.0, 0.0);
        }
        fft.inv(k, x, row, t);
        Y::put(x, row, t);
      }
    }
  };
  if constexpr (FWD) rows();
  else lines();
  __syncthreads();
  if constexpr (FWD) lines();
  else rows();
}

template <int NX, int NY, bool FWD>
static hipError_t launch_xyplane(const FFTCtx &c, int nf, const RealSet &re, const FieldSet &q, int prune) {
  constexpr PassShape s = plane_shape(NX, NY);
  static_assert(s.lines * Line<NX, FFTCfgMix<NX>>::T == (int)kRowBound, "a line of every T lanes");
  allow_lds(k_xyplane<NX, NY, FWD>, s.lds);
  GHX_LAUNCH_CHECK((k_xyplane<NX, NY, FWD>), s, kRowBound, 1, false);
  hipLaunchKernelGGL((k_xyplane<NX, NY, FWD>), dim3(c.gk.nz, nf), dim3(s.block), s.lds, c.stream, re, q, c.gk, c.tw_x, c.tw_y, prune);
  return hipGetLastError();
}
template <int NX, bool FWD>
static hipError_t plane_y(const FFTCtx &c, int nf, const RealSet &re, const FieldSet &q, int prune) {
  switch (c.gk.ny) {
#define GHX_CASE(n_) case n_: return launch_xyplane<NX, n_, FWD>(c, nf, re, q, prune);
    GHX_PLANE_SIZES(GHX_CASE)
#undef GHX_CASE
  default: return hipErrorInvalidValue;
  }
}
template <bool FWD>
static hipError_t plane_x(const FFTCtx &c, int nf, const RealSet &re, const FieldSet &q, int prune) {
  switch (c.gk.nx) {
#define GHX_CASE(n_) case n_: return plane_y<n_, FWD>(c, nf, re, q, prune);
    GHX_PLANE_SIZES(GHX_CASE)
#undef GHX_CASE
  default: return hipErrorInvalidValue;
  }
}
bool xyplane(const FFTCtx &c) {
  return plane_size(c.gk.nx) && plane_size(c.gk.ny) && use_x2(c.gk.nx) &&
         takes_plane(c.gk.nx, c.gk.ny, max_lds());
}
hipError_t xyplane_fwd(const FFTCtx &c, int nf, const double *const *in, const FieldSet &q) {
  RealSet rs;
  for (int f = 0; f < nf; ++f) rs.p[f] = const_cast<double *>(in[f]);
  return plane_x<true>(c, nf, rs, q, 0);
}
hipError_t xyplane_inv(const FFTCtx &c, int nf, const FieldSet &q, double *const *out, int prune) {
  RealSet rs;
  for (int f = 0; f < nf; ++f) rs.p[f] = out[f];
  return plane_x<false>(c, nf, rs, q, prune);
}
#endif

#if GHX_PART == 7
hipError_t xcross(const FFTCtx &c, int mode, const FieldSet &in, const FieldSet &out, int prune) {
  (void)mode;
  const GridK &g = c.gk;
  if (g.nx % 2) return hipErrorInvalidValue;
  const long nrows = (long)g.nz * g.ny;
  const int nxp = p_row(g);
  if (use_x2(g.nx)) {
    switch (g.nx) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    constexpr int T = FFTCfg<n_>::T;                                                        \
    const PassShape s = row_shape(T, lds_line_stride(n_), max_lds(), nrows * c.batch);                              \
    const int rpb = s.lines; const size_t lds = s.lds;                          \
    const dim3 gr((unsigned)((nrows + rpb - 1) / rpb), c.batch), bl(rpb * T);                      \
    GHX_LAUNCH_CHECK((k_xcross2<n_>), s, kRowBound, T, false); hipLaunchKernelGGL((k_xcross2<n_>), gr, bl, lds, c.stream, in, out, g, nxp, c.tw_x, kx_in(c, prune), kx_out(c, prune), prune_word(c, prune));                                                                 \
    return hipGetLastError();                                                               \
  }
      GHX_X2_SIZES(GHX_CASE)
#undef GHX_CASE
      default:
        break;
    }
  }
  switch (g.nx / 2) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    constexpr int T = FFTCfgLow<n_>::T;                                                     \
    const PassShape s = row_shape(T, lds_line_stride(n_), max_lds(), nrows * c.batch);                              \
    const int rpb = s.lines; const size_t lds = s.lds;                          \
    const dim3 gr((unsigned)((nrows + rpb - 1) / rpb), c.batch), bl(rpb * T);               \
    switch (tile_want("GHX_XV", 1)) {                                                       \
    case 4: GHX_LAUNCH_CHECK((k_xcross<n_, 2, 1>), s, kRowBound, T, false); hipLaunchKernelGGL((k_xcross<n_, 2, 1>), gr, bl, lds, c.stream, in, out, g, nxp, c.tw_xh, c.tw_x, kx_in(c, prune), kx_out(c, prune), prune_word(c, prune)); break; \
    /* 3 * 2^k rows: one wave per SIMD leaves the registers to hold the six */ \
    /* fields without scratch (7.5% faster on the ensemble's 48^3 and 96^3) */ \
    default: GHX_LAUNCH_CHECK((k_xcross<n_, (n_ % 3 == 0) ? 1 : 2, 0>), s, kRowBound, T, false); hipLaunchKernelGGL((k_xcross<n_, (n_ % 3 == 0) ? 1 : 2, 0>), gr, bl, lds, c.stream, in, out, g, nxp, c.tw_xh, c.tw_x, kx_in(c, prune), kx_out(c, prune), prune_word(c, prune)); break; \
    }                                                                                       \
    break;                                                                                  \
  }
    GHX_SIZES(GHX_CASE)
#undef GHX_CASE
  default:
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
#endif

}  // namespace ghx

#if GHX_PART == 8
namespace ghx {
hipError_t xdot(const FFTCtx &c, const FieldSet &in, const FieldSet &out, int prune) {
  const GridK &g = c.gk;
  if (g.nx % 2) return hipErrorInvalidValue;
  const long nrows = (long)g.nz * g.ny;
  const int nxp = p_row(g);
  if (use_x2(g.nx)) {
    switch (g.nx) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    constexpr int T = FFTCfg<n_>::T;                                                        \
    const PassShape s = row_shape(T, lds_line_stride(n_), max_lds(), nrows);                                        \
    const int rpb = s.lines; const size_t lds = s.lds;                          \
    const dim3 gr((unsigned)((nrows + rpb - 1) / rpb)), bl(rpb * T);                      \
    GHX_LAUNCH_CHECK((k_xdot2<n_>), s, kRowBound, T, false); hipLaunchKernelGGL((k_xdot2<n_>), gr, bl, lds, c.stream, in, out, g, nxp, c.tw_x, kx_in(c, prune), kx_out(c, prune), prune_word(c, prune));                                                                 \
    return hipGetLastError();                                                               \
  }
      GHX_X2_SIZES(GHX_CASE)
#undef GHX_CASE
      default:
        break;
    }
  }
  switch (g.nx / 2) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    constexpr int T = FFTCfgLow<n_>::T;                                                     \
    const PassShape s = row_shape(T, lds_line_stride(n_), max_lds(), nrows);                                        \
    const int rpb = s.lines; const size_t lds = s.lds;                          \
    GHX_LAUNCH_CHECK((k_xdot<n_>), s, kRowBound, T, false); hipLaunchKernelGGL((k_xdot<n_>), dim3((unsigned)((nrows + rpb - 1) / rpb)), dim3(rpb * T), lds, c.stream, in, out, g, nxp, c.tw_xh, c.tw_x, kx_in(c, prune), kx_out(c, prune), prune_word(c, prune)); \
    break;                                                                                  \
  }
    GHX_SIZES(GHX_CASE)
#undef GHX_CASE
  default:
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t zfwd_rk_bouss(const FFTCtx &c, const FieldSet &in, const BoussRKParams &rk, int prune) {
  const GridK &g = c.gk;
  // Up to kSmallLines at any length (63 against 78 us for 2112 lines of 512
  // points, 115 against 196 of 1024), and beyond on power-of-two lines of 32 to
  // 256 points: 48 -> 26 us at 128^3, 207 -> 169 at 256^3, 113 -> 83 at 256 x 256 x 128
  // (but 37 -> 47 at 192 x 192 x 96)
  if ((z_lines(c) <= kSmallLines || (g.nz >= 32 && g.nz <= 256 && (g.nz & (g.nz - 1)) == 0)) &&
      takes_zrk(zrk_groups(2), lds_line_stride(g.nz), max_lds())) {
    ZUpdate u{};
    u.dt = rk.dt; u.rmp = rk.rmp; u.nu = rk.nu; u.mu = rk.kappa; u.om2 = rk.om2; u.xmom = rk.xmom; u.xtemp = rk.xtemp;
    u.fline = rk.fline;
    for (int k = 0; k < 4; ++k) { u.v[k] = rk.v[k]; u.c[k] = rk.c[k]; u.f[k] = rk.f[k]; u.out[k] = rk.out[k]; }
    switch (g.nz) {
#define GHX_CASE(n_) case n_: return launch_zrk<n_, 2, FFTCfgMix<n_>>(c, in, u, prune, 1);
      GHX_SIZES(GHX_CASE)
#undef GHX_CASE
    default: return hipErrorInvalidValue;
    }
  }
  // 2 lines of 64 lanes and more (509 -> 455 us at 256 x 256 x 512)
  switch (g.nz) {
#define GHX_CASE(n_)                                                                        \
  case n_: {                                                                                \
    constexpr int T = FFTCfg<n_>::T;                                                        \
    const PassShape s = tile_shape(T, lds_line_stride(n_) + n_, g.ny, tile_want("GHX_LZ", T >= 64 ? 2 : tile_default(T, 4)), max_lds());              \
    const int L = s.lines; const size_t lds = s.lds;                     \
    dim3 grid((g.ny + L - 1) / L, g.nxh);                                                   \
    using Cfg = ZBoussCfg<n_>;                                                              \
    allow_lds((k_zfwd_rk_bouss<n_, Cfg>), lds);                                                    \
    GHX_LAUNCH_CHECK((k_zfwd_rk_bouss<n_, Cfg>), s, kTileBound, T, true); hipLaunchKernelGGL((k_zfwd_rk_bouss<n_, Cfg>), grid, dim3(L * T), lds, c.stream, in, g, c.tw_z, rk, prune); \
    break;                                                                                  \
  }
    GHX_SIZES(GHX_CASE)
#undef GHX_CASE
  default:
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
}  // namespace ghx
#endif
