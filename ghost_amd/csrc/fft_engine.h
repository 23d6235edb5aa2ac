// fft_engine.h -- register-resident Stockham line FFT for gfx950 (FP64 complex).
//
// A line of N complex points is held by T = N/E lanes, E points per lane:
// lane t holds elements t + T*m (m = 0..E-1).  Every Stockham stage reads
// exactly that set, so a stage is: E/R radix-R butterflies in registers, then
// an exchange through a padded LDS line buffer.  The last stage needs no
// exchange: its outputs land back in the same register slots in natural order.
// For N = 512 (E = 8, radix 8^3) a line is one 64-wide wavefront.
//
// Transform convention (FFTW's, which GHOST uses): DIR = -1 forward,
// DIR = +1 inverse, both unnormalised.
#pragma once
#include <type_traits>
#include "ghx_common.h"

// LDS padding: one spare slot every 8 complex points keeps the stride-R
// butterfly writes of the first stages on distinct banks.
GHX_DEV int lds_pad(int i) { return i + (i >> 3); }
__host__ __device__ constexpr int lds_line_stride(int n) { return n + (n >> 3) + 1; }

// ---------------------------------------------------------------------------
// Per-size schedule: E points per lane and the radix of each stage.
// ---------------------------------------------------------------------------
template <int N> struct FFTCfg;
#define GHX_FFTCFG(N_, E_, NS_, ...)                                    \
  template <> struct FFTCfg<N_> {                                       \
    static constexpr int E = E_;                                        \
    static constexpr int NS = NS_;                                      \
    static constexpr int T = N_ / E_;                                   \
    GHX_DEV static constexpr int radix(int s) {                         \
      constexpr int r[] = {__VA_ARGS__};                                \
      return r[s];                                                      \
    }                                                                   \
  };
GHX_FFTCFG(1, 1, 0, 1)
GHX_FFTCFG(2, 2, 1, 2)
GHX_FFTCFG(3, 3, 1, 3)
GHX_FFTCFG(4, 4, 1, 4)
GHX_FFTCFG(5, 5, 1, 5)
GHX_FFTCFG(6, 6, 2, 3, 2)
GHX_FFTCFG(8, 8, 1, 8)
GHX_FFTCFG(10, 10, 2, 5, 2)
GHX_FFTCFG(12, 12, 2, 3, 4)
GHX_FFTCFG(16, 8, 2, 2, 8)
GHX_FFTCFG(20, 20, 2, 5, 4)
GHX_FFTCFG(24, 6, 3, 6, 2, 2)
GHX_FFTCFG(32, 8, 2, 4, 8)
GHX_FFTCFG(40, 40, 2, 5, 8)
GHX_FFTCFG(48, 6, 4, 6, 2, 2, 2)
GHX_FFTCFG(64, 8, 2, 8, 8)
GHX_FFTCFG(80, 40, 3, 5, 2, 8)
GHX_FFTCFG(96, 6, 5, 6, 2, 2, 2, 2)
GHX_FFTCFG(128, 8, 3, 2, 8, 8)
GHX_FFTCFG(160, 40, 3, 5, 4, 8)
GHX_FFTCFG(192, 6, 6, 6, 2, 2, 2, 2, 2)
GHX_FFTCFG(256, 8, 3, 4, 8, 8)
GHX_FFTCFG(384, 6, 7, 6, 2, 2, 2, 2, 2, 2)
GHX_FFTCFG(512, 8, 3, 8, 8, 8)
GHX_FFTCFG(768, 24, 4, 3, 4, 8, 8)
GHX_FFTCFG(1024, 8, 4, 2, 8, 8, 8)

// Low-register schedules (4 points per lane) for kernels that keep several
// fields live at once (the fused x pass holds six); other sizes fall back to
// the default schedule.
template <int N> struct FFTCfgLow : FFTCfg<N> {};
#define GHX_FFTCFGLOW(N_, E_, NS_, ...)                                 \
  template <> struct FFTCfgLow<N_> {                                    \
    static constexpr int E = E_;                                        \
    static constexpr int NS = NS_;                                      \
    static constexpr int T = N_ / E_;                                   \
    GHX_DEV static constexpr int radix(int s) {                         \
      constexpr int r[] = {__VA_ARGS__};                                \
      return r[s];                                                      \
    }                                                                   \
  };
GHX_FFTCFGLOW(32, 4, 3, 2, 4, 4)
GHX_FFTCFGLOW(64, 4, 3, 4, 4, 4)
GHX_FFTCFGLOW(128, 4, 4, 2, 4, 4, 4)
GHX_FFTCFGLOW(256, 4, 4, 4, 4, 4, 4)
GHX_FFTCFGLOW(512, 4, 5, 2, 4, 4, 4, 4)
#undef GHX_FFTCFGLOW

// Wide schedules (16 points per lane, half the lanes per line) for passes
// whose blocks should hold more lines with fewer lanes.
template <int N> struct FFTCfgWide : FFTCfg<N> {};
template <> struct FFTCfgWide<512> {
  static constexpr int E = 16;
  static constexpr int NS = 3;
  static constexpr int T = 512 / 16;
  GHX_DEV static constexpr int radix(int) { return 8; }
};

// 12 points per lane for the 3 * 2^k lines, for passes that keep one field live
// and wait on memory more than on their exchanges (the y passes, the one-field
// z inverses).  The others take the mixed stages (MixFFT).
template <int N> struct FFTCfgMid : FFTCfg<N> {};
#define GHX_FFTCFGMID(N_, NS_, ...)                                     \
  template <> struct FFTCfgMid<N_> {                                    \
    static constexpr int E = 12;                                        \
    static constexpr int NS = NS_;                                      \
    static constexpr int T = N_ / 12;                                   \
    GHX_DEV static constexpr int radix(int s) {                         \
      constexpr int r[] = {__VA_ARGS__};                                \
      return r[s];                                                      \
    }                                                                   \
  };
GHX_FFTCFGMID(96, 3, 12, 4, 2)
GHX_FFTCFGMID(192, 3, 12, 4, 4)
GHX_FFTCFGMID(384, 4, 12, 4, 4, 2)
#undef GHX_FFTCFGMID
#undef GHX_FFTCFG

// ---------------------------------------------------------------------------
// Small DFTs in registers, sign DIR.
// ---------------------------------------------------------------------------
template <int R, int DIR> struct SmallDFT;

template <int DIR> struct SmallDFT<1, DIR> {
  GHX_DEV static void run(cplx *) {}
};
template <int DIR> struct SmallDFT<2, DIR> {
  GHX_DEV static void run(cplx *v) {
    cplx a = c_add(v[0], v[1]), b = c_sub(v[0], v[1]);
    v[0] = a; v[1] = b;
  }
};
template <int DIR> struct SmallDFT<3, DIR> {
  GHX_DEV static void run(cplx *v) {
    const double s3 = 0.86602540378443864676;
    cplx t = c_add(v[1], v[2]), d = c_sub(v[1], v[2]);
    cplx m = c_sub(v[0], c_scale(t, 0.5));
    cplx e = c_mul_si<DIR>(c_scale(d, s3));
    v[0] = c_add(v[0], t);
    v[1] = c_add(m, e);
    v[2] = c_sub(m, e);
  }
};
template <int DIR> struct SmallDFT<4, DIR> {
  GHX_DEV static void run(cplx *v) {
    cplx a0 = c_add(v[0], v[2]), a1 = c_sub(v[0], v[2]);
    cplx a2 = c_add(v[1], v[3]), a3 = c_mul_si<DIR>(c_sub(v[1], v[3]));
    v[0] = c_add(a0, a2); v[2] = c_sub(a0, a2);
    v[1] = c_add(a1, a3); v[3] = c_sub(a1, a3);
  }
};
template <int DIR> struct SmallDFT<5, DIR> {
  GHX_DEV static void run(cplx *v) {
    // Winograd-style radix 5 with c1 = cos(2pi/5), c2 = cos(4pi/5), s1, s2 sines.
    const double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
    const double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;
    cplx t1 = c_add(v[1], v[4]), t2 = c_add(v[2], v[3]);
    cplx t3 = c_sub(v[1], v[4]), t4 = c_sub(v[2], v[3]);
    cplx a1 = c_add(v[0], c_add(c_scale(t1, c1), c_scale(t2, c2)));
    cplx a2 = c_add(v[0], c_add(c_scale(t1, c2), c_scale(t2, c1)));
    cplx b1 = c_mul_si<DIR>(c_add(c_scale(t3, s1), c_scale(t4, s2)));
    cplx b2 = c_mul_si<DIR>(c_sub(c_scale(t3, s2), c_scale(t4, s1)));
    v[0] = c_add(v[0], c_add(t1, t2));
    v[1] = c_add(a1, b1); v[4] = c_sub(a1, b1);
    v[2] = c_add(a2, b2); v[3] = c_sub(a2, b2);
  }
};
// 6 = 3 x 2 and 12 = 3 x 4 by the prime-factor (Good-Thomas) maps, which need
// no twiddles between the factors: with n = 2a + 3b, k = 4c + 3d (mod 6),
// nk = 2ac + 3bd; with n = 4a + 3b, k = 4c + 9d (mod 12), nk = 4ac + 3bd.
template <int DIR> struct SmallDFT<6, DIR> {
  GHX_DEV static void run(cplx *v) {
    cplx x[2][3];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int a = 0; a < 3; ++a) x[b][a] = v[(2 * a + 3 * b) % 6];
      SmallDFT<3, DIR>::run(x[b]);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      v[(4 * c) % 6] = c_add(x[0][c], x[1][c]);
      v[(4 * c + 3) % 6] = c_sub(x[0][c], x[1][c]);
    }
  }
};
template <int DIR> struct SmallDFT<12, DIR> {
  GHX_DEV static void run(cplx *v) {
    cplx x[4][3];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
#pragma unroll
      for (int a = 0; a < 3; ++a) x[b][a] = v[(4 * a + 3 * b) % 12];
      SmallDFT<3, DIR>::run(x[b]);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      cplx y[4] = {x[0][c], x[1][c], x[2][c], x[3][c]};
      SmallDFT<4, DIR>::run(y);
#pragma unroll
      for (int d = 0; d < 4; ++d) v[(4 * c + 9 * d) % 12] = y[d];
    }
  }
};
template <int DIR> struct SmallDFT<8, DIR> {
  GHX_DEV static void run(cplx *v) {
    const double r2 = 0.70710678118654752440;
    cplx e[4] = {v[0], v[2], v[4], v[6]};
    cplx o[4] = {v[1], v[3], v[5], v[7]};
    SmallDFT<4, DIR>::run(e);
    SmallDFT<4, DIR>::run(o);
    // W8 = exp(DIR*2 pi i/8) = (1 + DIR i)/sqrt 2
    cplx o1 = c_scale(c_add(o[1], c_mul_si<DIR>(o[1])), r2);
    cplx o2 = c_mul_si<DIR>(o[2]);
    cplx o3 = c_mul_si<DIR>(c_scale(c_add(o[3], c_mul_si<DIR>(o[3])), r2));
    v[0] = c_add(e[0], o[0]); v[4] = c_sub(e[0], o[0]);
    v[1] = c_add(e[1], o1);   v[5] = c_sub(e[1], o1);
    v[2] = c_add(e[2], o2);   v[6] = c_sub(e[2], o2);
    v[3] = c_add(e[3], o3);   v[7] = c_sub(e[3], o3);
  }
};

// ---------------------------------------------------------------------------
// Twiddle powers w^1..w^(R-1) from one table load by a product tree of depth
// <= 3 (rounding error of a few ulp), instead of R-1 table loads.
// ---------------------------------------------------------------------------
template <int R> GHX_DEV void tw_powers(cplx w1, cplx *w) {
  w[1] = w1;
  if constexpr (R > 2) w[2] = c_mul(w1, w1);
  if constexpr (R > 3) w[3] = c_mul(w[2], w1);
  if constexpr (R > 4) w[4] = c_mul(w[2], w[2]);
  if constexpr (R > 5) w[5] = c_mul(w[4], w1);
  if constexpr (R > 6) w[6] = c_mul(w[3], w[3]);
  if constexpr (R > 7) w[7] = c_mul(w[4], w[3]);
}

// The same with more of the powers read, for the lines of 3 * 2^k points: w1 and
// w3 for radix 8, w1 and w2 for radix 4, w1 to w3 for radix 6, so that no power
// is further than two products from correctly rounded roots.  RMS relative error
// of one line of random points in units of 1e-16, radix-3 and radix-2 stages
// with every twiddle from the table | one root and the tree above | these: the
// mixed stages' inverse 1.55 | 1.80 | 1.50 (24 points), 1.70 | 2.40 | 1.63 (48),
// 1.86 | 2.17 | 1.84 (96), 2.01 | 2.73 | 1.90 (192), 2.13 | 3.22 | 2.12 (384);
// their forward 1.55 | 2.31 | 1.41, 1.70 | 2.11 | 1.60, 1.86 | 2.29 | 1.69, 2.01
// | 2.77 | 1.92, 2.13 | 3.09 | 2.09; 12 points per lane 1.86 | 1.87 | 1.69 (96),
// 2.01 | 2.13 | 1.84 (192), 2.13 | 2.26 | 1.99 (384).  (w3 of radix 4 read as
// well costs a wave per SIMD: MHD z inverse 23.7 -> 26.5 us at 96^3.)
// FULL: every power read, for passes with registers to spare.
template <int R, bool FULL = false> constexpr int tw_nroots() { return FULL ? R - 1 : R == 6 ? 3 : R == 4 || R == 8 ? 2 : 1; }
// the power that the r-th root read is
template <int R, bool FULL = false> constexpr int tw_power(int r) { return !FULL && R == 8 && r == 1 ? 3 : r + 1; }
template <int R, int M> GHX_DEV void tw_powers(const cplx (&p)[M], cplx *w) {
  w[1] = p[0];
  if constexpr (M == R - 1) {
#pragma unroll
    for (int r = 2; r < R; ++r) w[r] = p[r - 1];
  } else if constexpr (M == 1) {
    tw_powers<R>(p[0], w);
  } else {
    static_assert(M == tw_nroots<R>(), "the roots of the 3 * 2^k lines");
    if constexpr (R == 4) w[2] = p[1], w[3] = c_mul(p[0], p[1]);
    if constexpr (R == 6) w[2] = p[1], w[3] = p[2], w[4] = c_mul(p[1], p[1]), w[5] = c_mul(p[1], p[2]);
    if constexpr (R == 8) {
      w[2] = c_mul(p[0], p[0]);
      w[3] = p[1];
      w[4] = c_mul(p[0], p[1]);
      w[5] = c_mul(w[2], p[1]);
      w[6] = c_mul(p[1], p[1]);
      w[7] = c_mul(w[4], p[1]);
    }
  }
}

// A schedule Cfg whose stages read more roots than its length asks for: the
// tw_nroots of the 3 * 2^k lines, or with FULL every power.
template <typename Cfg, bool FULL> struct FFTCfgRoots : Cfg {};
template <typename Cfg> struct cfg_roots { static constexpr int value = 0; };
template <typename Cfg, bool FULL> struct cfg_roots<FFTCfgRoots<Cfg, FULL>> { static constexpr int value = FULL ? 2 : 1; };

// ---------------------------------------------------------------------------
// Synchronisation of one line's LDS exchange.  A line of T <= 64 lanes lives
// inside one wavefront (T is a power of two and blocks are whole lines), so
// ordering the wave's own LDS traffic is enough and the other waves of the
// block run on; longer lines need the block barrier.
// ---------------------------------------------------------------------------
template <int T> GHX_DEV void line_sync() {
  if constexpr (T <= 64) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Twiddle sources for the stages.  TwTable reads the root of each butterfly
// from the forward table when the stage runs; TwCache holds the roots of one
// lane for every stage of one schedule in registers, loaded once, for kernels
// that run many transforms of the same length per lane.
// ---------------------------------------------------------------------------
// A butterfly reads one root, more on the lines of 3 * 2^k points and on FFTCfgRoots.
template <int N, int R, typename Cfg> constexpr int line_nroots() {
  return (N % 3 == 0 && N >= 24) || cfg_roots<Cfg>::value > 0 ? tw_nroots<R, cfg_roots<Cfg>::value == 2>() : 1;
}
template <int N, int R, typename Cfg> constexpr int line_power(int r) {
  return line_nroots<N, R, Cfg>() > 1 ? tw_power<R, cfg_roots<Cfg>::value == 2>(r) : 1;
}
struct TwTable {
  const cplx *p;
  template <int S> GHX_DEV cplx root(int, int r, int idx) const { (void)r; return p[idx]; }
};

template <int N, typename Cfg = FFTCfg<N>> struct TwCache {
  static constexpr int NS = Cfg::NS, E = Cfg::E, T = Cfg::T;
  cplx w[NS > 0 ? NS : 1][E];
  template <int S, int Ns> GHX_DEV void fill(const cplx *tw, int t) {
    if constexpr (S < NS) {
      constexpr int R = Cfg::radix(S), Q = E / R, M = line_nroots<N, R, Cfg>();
      if constexpr (Ns > 1) {
        constexpr int tws = N / (Ns * R);
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
          for (int r = 0; r < M; ++r) w[S][q * M + r] = tw[((t + q * T) % Ns) * line_power<N, R, Cfg>(r) * tws];
      }
      fill<S + 1, Ns * R>(tw, t);
    }
  }
  GHX_DEV void load(const cplx *tw, int t) { fill<0, 1>(tw, t); }
  template <int S> GHX_DEV cplx root(int q, int r, int) const {
    return w[S][q * line_nroots<N, Cfg::radix(S), Cfg>() + r];
  }
};

// ---------------------------------------------------------------------------
// The line transform.
// ---------------------------------------------------------------------------
template <int N, int DIR, typename Cfg = FFTCfg<N>> struct LineFFT {
  using C = Cfg;
  static constexpr int E = C::E;
  static constexpr int T = C::T;

  // One Stockham stage (radix R, Ns = product of earlier radices).  If LAST,
  // the outputs stay in v; otherwise they are written to the LDS line buffer
  // and v is reloaded from it.
  template <int S, int NsS, typename TW>
  GHX_DEV static void stages(cplx (&v)[E], cplx *buf, int t, const TW &tw) {
    if constexpr (S < C::NS) {
      constexpr int R = C::radix(S);
      constexpr int Q = E / R;
      constexpr int Ns = NsS;
      constexpr bool LAST = (S == C::NS - 1);
      static_assert(E % R == 0, "radix must divide points per lane");
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int j = t + q * T;
        cplx u[R];
#pragma unroll
        for (int r = 0; r < R; ++r) u[r] = v[q + r * Q];
        if constexpr (Ns > 1) {
          const int k = j % Ns;
          constexpr int tws = N / (Ns * R);
          cplx w[R];
          constexpr int M = line_nroots<N, R, Cfg>();
          cplx p[M];
#pragma unroll
          for (int r = 0; r < M; ++r) {
            const cplx x = tw.template root<S>(q, r, k * line_power<N, R, Cfg>(r) * tws);
            p[r] = DIR < 0 ? x : c_conj(x);
          }
          tw_powers<R, M>(p, w);
#pragma unroll
          for (int r = 1; r < R; ++r) u[r] = c_mul(u[r], w[r]);
        }
        SmallDFT<R, DIR>::run(u);
        if constexpr (LAST) {
#pragma unroll
          for (int r = 0; r < R; ++r) v[q + r * Q] = u[r];
        } else {
          const int base = (j / Ns) * Ns * R + (j % Ns);
#pragma unroll
          for (int r = 0; r < R; ++r) buf[lds_pad(base + r * Ns)] = u[r];
        }
      }
      if constexpr (!LAST) {
        line_sync<T>();
#pragma unroll
        for (int m = 0; m < E; ++m) v[m] = buf[lds_pad(t + T * m)];
        line_sync<T>();
        stages<S + 1, Ns * R, TW>(v, buf, t, tw);
      }
    }
  }

  // v holds x[t + T m] on entry and X[t + T m] on exit.  buf is this line's
  // LDS buffer (lds_line_stride(N) slots), used by this line only.  Every
  // thread of the block must call this (lines longer than a wavefront use
  // block barriers).
  GHX_DEV static void run(cplx (&v)[E], cplx *buf, int t, const cplx *tw) {
    stages<0, 1, TwTable>(v, buf, t, TwTable{tw});
  }
  // the same with the stage roots held in registers (TwCache<N, Cfg> of the
  // forward table, loaded by this lane)
  GHX_DEV static void run(cplx (&v)[E], cplx *buf, int t, const TwCache<N, Cfg> &tw) {
    stages<0, 1, TwCache<N, Cfg>>(v, buf, t, tw);
  }
};

// ---------------------------------------------------------------------------
// Lines of N = 3 * 2^k points (24 .. 384) in two or three stages of radix 6
// and 8 or 4, instead of radix 6 and then 2, 2, ..: the lanes per stage differ.
// The radix-6 stage uses all T = N / 6 lanes of the line with 6 points each,
// the others A = N / 8 = 3/4 T of them with 8 points each, so a line takes one
// or two LDS exchanges where the 6-point schedules take two to six.  The
// inverse starts with radix 6, the forward ends with it: the wavenumber side
// is held as x[t + T m] (m < 6) by every lane, the other side as x[t + A m]
// (m < 8) by the lanes t < A, and a pass that does both needs no exchange to
// get from one to the other.  Measured, 6-point schedule -> mixed stages, us: X
// cross 1084 -> 729 at 384^3, 125 -> 100 at 192^3, 24.7 -> 21.6 at 96^3, 11.6 ->
// 9.0 at 48^3, 10.5 -> 8.2 at 24^3; X dot 116 -> 88 at 384 x 192 x 96; three
// interleaved x inverses 606 -> 440 at 384^3; one field's x inverse 200 -> 163,
// x forward 196 -> 170 and z forward 266 -> 238 at 384^3; curl z inverse 391 ->
// 325 at 384^3, 54 -> 46 at 192^3; MHD z inverse 97 -> 83, HD update 52 -> 47 at
// 192^3, 57 -> 32 at 96 x 96 x 384.
// ---------------------------------------------------------------------------
template <int N> struct MixCfg;  // radices of the 8-point stages, in the inverse's order (1: no stage)
template <> struct MixCfg<24> { static constexpr int R1 = 4, R2 = 1; };
template <> struct MixCfg<48> { static constexpr int R1 = 8, R2 = 1; };
template <> struct MixCfg<96> { static constexpr int R1 = 4, R2 = 4; };
template <> struct MixCfg<192> { static constexpr int R1 = 8, R2 = 4; };
template <> struct MixCfg<384> { static constexpr int R1 = 8, R2 = 8; };

template <int N, int DIR, bool FULL = false> struct MixFFT {
  using C = MixCfg<N>;
  static constexpr int T = N / 6, A = N / 8;
  static_assert(6 * C::R1 * C::R2 == N && T <= 64, "a line lives in one wavefront");

  // the stage's roots of this lane, tw_nroots of each butterfly
  template <int R, int E> struct Stage {
    cplx w[E / R][tw_nroots<R, FULL>()];
    template <int Ns, int L> GHX_DEV void load(const cplx *tw, int t) {
#pragma unroll
      for (int q = 0; q < E / R; ++q)
#pragma unroll
        for (int r = 0; r < tw_nroots<R, FULL>(); ++r) w[q][r] = tw[((t + q * L) % Ns) * tw_power<R, FULL>(r) * (N / (Ns * R))];
    }
  };
  template <int R, bool TWIDDLE, int E> GHX_DEV static void butterflies(cplx (&v)[E], const Stage<R, E> *st) {
    constexpr int Q = E / R;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      cplx u[R];
#pragma unroll
      for (int r = 0; r < R; ++r) u[r] = v[q + r * Q];
      if constexpr (TWIDDLE) {
        cplx w[R], p[tw_nroots<R, FULL>()];
#pragma unroll
        for (int r = 0; r < tw_nroots<R, FULL>(); ++r) p[r] = DIR < 0 ? st->w[q][r] : c_conj(st->w[q][r]);
        tw_powers<R, tw_nroots<R, FULL>()>(p, w);
#pragma unroll
        for (int r = 1; r < R; ++r) u[r] = c_mul(u[r], w[r]);
      }
      SmallDFT<R, DIR>::run(u);
#pragma unroll
      for (int r = 0; r < R; ++r) v[q + r * Q] = u[r];
    }
  }
  template <int R, int Ns, int L, int E> GHX_DEV static void put(const cplx (&v)[E], cplx *buf, int t) {
    constexpr int Q = E / R;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int j = t + q * L, base = (j / Ns) * Ns * R + (j % Ns);
#pragma unroll
      for (int r = 0; r < R; ++r) buf[lds_pad(base + r * Ns)] = v[q + r * Q];
    }
  }
  template <int L, int E> GHX_DEV static void get(cplx (&v)[E], const cplx *buf, int t) {
#pragma unroll
    for (int m = 0; m < E; ++m) v[m] = buf[lds_pad(t + L * m)];
  }

  struct None {};
  // wavenumbers in (t + T m) -> samples out (t + A m, lanes t < A)
  struct Inv {
    Stage<C::R1, 8> a;
    typename std::conditional<(C::R2 > 1), Stage<C::R2, 8>, None>::type b;
    GHX_DEV void load(const cplx *tw, int t) {
      a.template load<6, A>(tw, t);
      if constexpr (C::R2 > 1) b.template load<6 * C::R1, A>(tw, t);
    }
    GHX_DEV void run(cplx (&in)[6], cplx (&out)[8], cplx *buf, int t) const {
      butterflies<6, false, 6>(in, nullptr);
      put<6, 1, T, 6>(in, buf, t);
      line_sync<T>();
      if (t < A) {
        get<A, 8>(out, buf, t);
        butterflies<C::R1, true, 8>(out, &a);
      }
      line_sync<T>();
      if constexpr (C::R2 > 1) {
        if (t < A) put<C::R1, 6, A, 8>(out, buf, t);
        line_sync<T>();
        if (t < A) {
          get<A, 8>(out, buf, t);
          butterflies<C::R2, true, 8>(out, &b);
        }
        line_sync<T>();
      }
    }
  };
  // samples in (t + A m, lanes t < A) -> wavenumbers out (t + T m)
  struct Fwd {
    typename std::conditional<(C::R2 > 1), Stage<C::R1, 8>, None>::type b;
    Stage<6, 6> c;
    GHX_DEV void load(const cplx *tw, int t) {
      if constexpr (C::R2 > 1) b.template load<C::R2, A>(tw, t);
      c.template load<N / 6, T>(tw, t);
    }
    GHX_DEV void run(cplx (&in)[8], cplx (&out)[6], cplx *buf, int t) const {
      if constexpr (C::R2 > 1) {
        if (t < A) {
          butterflies<C::R2, false, 8>(in, nullptr);
          put<C::R2, 1, A, 8>(in, buf, t);
        }
        line_sync<T>();
        if (t < A) {
          get<A, 8>(in, buf, t);
          butterflies<C::R1, true, 8>(in, &b);
        }
        line_sync<T>();
        if (t < A) put<C::R1, C::R2, A, 8>(in, buf, t);
      } else if (t < A) {
        butterflies<C::R1, false, 8>(in, nullptr);
        put<C::R1, 1, A, 8>(in, buf, t);
      }
      line_sync<T>();
      get<T, 6>(out, buf, t);
      line_sync<T>();
      butterflies<6, true, 6>(out, &c);
    }
  };
};

// One lane's part of a line's transforms in either direction, with KE points
// on the wavenumber side (k = t + T m, every lane) and SE on the sample side
// (n = t + A m, in the lanes with live(t)): LineFFT of a schedule Cfg, one
// layout on both sides, or MixFFT for FFTCfgMixed.
constexpr bool mix_length(int n) { return n == 24 || n == 48 || n == 96 || n == 192 || n == 384; }
template <int N> struct FFTCfgMixed {
  static constexpr int E = 6, T = N / 6;
};
template <int N>
using FFTCfgMix = typename std::conditional<mix_length(N), FFTCfgMixed<N>, FFTCfg<N>>::type;

template <int N, typename Cfg = FFTCfg<N>> struct Line {
  static constexpr int T = Cfg::T, A = T, KE = Cfg::E, SE = Cfg::E;
  TwCache<N, Cfg> tw;
  GHX_DEV void load_inv(const cplx *w, int t) { tw.load(w, t); }
  GHX_DEV void load_fwd(const cplx *w, int t) { tw.load(w, t); }
  GHX_DEV void load_fwd_too(const cplx *, int) {}  // after load_inv: the same roots
  GHX_DEV static constexpr bool live(int) { return true; }
  GHX_DEV void inv(cplx (&k)[KE], cplx (&x)[SE], cplx *buf, int t) const {
#pragma unroll
    for (int m = 0; m < SE; ++m) x[m] = k[m];
    LineFFT<N, +1, Cfg>::run(x, buf, t, tw);
  }
  GHX_DEV void fwd(cplx (&x)[SE], cplx (&k)[KE], cplx *buf, int t) const {
#pragma unroll
    for (int m = 0; m < KE; ++m) k[m] = x[m];
    LineFFT<N, -1, Cfg>::run(k, buf, t, tw);
  }
  // samples to and from the line's LDS row
  GHX_DEV static void put(const cplx (&x)[SE], cplx *row, int t) {
#pragma unroll
    for (int m = 0; m < SE; ++m) row[lds_pad(t + T * m)] = x[m];
  }
  GHX_DEV static void get(cplx (&x)[SE], const cplx *row, int t) {
#pragma unroll
    for (int m = 0; m < SE; ++m) x[m] = row[lds_pad(t + T * m)];
  }
};
template <int N, bool FULL> struct MixLine {
  using I = MixFFT<N, +1, FULL>;
  using F = MixFFT<N, -1, FULL>;
  static constexpr int T = I::T, A = I::A, KE = 6, SE = 8;
  typename I::Inv wi;
  typename F::Fwd wf;
  GHX_DEV void load_inv(const cplx *w, int t) { wi.load(w, t); }
  GHX_DEV void load_fwd(const cplx *w, int t) { wf.load(w, t); }
  GHX_DEV void load_fwd_too(const cplx *w, int t) { wf.load(w, t); }
  GHX_DEV static bool live(int t) { return t < A; }
  GHX_DEV void inv(cplx (&k)[6], cplx (&x)[8], cplx *buf, int t) const { wi.run(k, x, buf, t); }
  GHX_DEV void fwd(cplx (&x)[8], cplx (&k)[6], cplx *buf, int t) const { wf.run(x, k, buf, t); }
  GHX_DEV static void put(const cplx (&x)[8], cplx *row, int t) {
    if (t < A) {
#pragma unroll
      for (int m = 0; m < 8; ++m) row[lds_pad(t + A * m)] = x[m];
    }
  }
  GHX_DEV static void get(cplx (&x)[8], const cplx *row, int t) {
    if (t < A) {
#pragma unroll
      for (int m = 0; m < 8; ++m) x[m] = row[lds_pad(t + A * m)];
    }
  }
};
template <int N> struct Line<N, FFTCfgMixed<N>> : MixLine<N, false> {};
template <int N, bool FULL> struct Line<N, FFTCfgRoots<FFTCfgMixed<N>, FULL>> : MixLine<N, FULL> {};
