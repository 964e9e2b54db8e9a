// cf_fft.hpp -- FP64 real transforms of N^3 lattices as three passes of short FFTs in
// LDS (the inverse of a small lattice takes the last two in one kernel, plane by plane),
// with the element-wise work around a transform folded into its passes.
//
// A block transforms FFT_CW = 8 neighbouring lines at once. In LDS element e of line l
// sits at [e][l], 16 bytes each, so eight lanes touch 128 contiguous bytes whatever the
// element stride of a stage: no bank conflicts in any radix. In memory the same eight
// lines are eight consecutive c of a row (passes along a and b: one 128-byte line per
// element) or eight rows (pass along c). There the lanes that read or write memory run
// along a row instead, eight 16-byte elements each, and the lines of an element are
// rotated in LDS by (e + e / M) mod 8 (M: the first stage's stride), so that neither
// consecutive elements nor consecutive frequencies share banks. (With lanes across the
// rows in memory too, every 16 bytes were a line of their own: 717 us for the complex-to-
// real pass of two N=384 fields.)
//
// The stages are decimation in frequency, in place: a butterfly reads its R elements and
// writes them back to the same slots, one barrier per stage, one buffer. The first stage
// reads global memory and the last writes it, so a pass of S stages makes S - 1 round
// trips through LDS. The last stage's results come in digit-reversed order, which costs
// nothing where every element is its own 128-byte line. Sizes with no prime factor above
// 7 are covered by radices 2 .. 8; the stage loop and its strides are run-time values
// (uniform), division by a stage's stride is a multiply and shift. Roots of unity come
// from a table of N (extended precision on the host), kept in LDS.
//
// What bounds it: memory. One pass over the half spectrum reads and writes it once; the
// library's passes along a and b took 0.70 and 0.78 ms at N=384 for two fields (1.8 GB
// of traffic each, 2.3-2.6 TB/s).
//
// Error against extended precision, N = 32 .. 1024: 2.2e-16 to 7.2e-16 relative (2-norm) in
// either direction; the library's 2.8e-16 to 1.1e-15, the larger at every size measured.
// Above N = 560 a block's lines and roots take more than half of a CU's LDS and one block of
// eight wavefronts runs there; still us for a forward transform, library / here: N=576 4006 / 2374,
// 640 5675 / 3081, 768 9893 / 5047, 972 22315 / 11370, 1024 22611 / 12462.
#pragma once

#include "cf_common.hpp"

namespace cf {

constexpr int FFT_CW = 8;         // lines per block
constexpr int FFT_MAX_STAGES = 6;
constexpr int FFT_MAX_N = 1024;

// Plan of one complex length n, read by the kernels (by value).
struct FftLen {
  int n = 0, stages = 0;
  int rad[FFT_MAX_STAGES] = {};
  int len[FFT_MAX_STAGES] = {};  // block length L of the stage
  int inv[FFT_MAX_STAGES] = {};  // ceil(2^20 / (L / R)): b / (L / R) = (b * inv) >> 20 for b < 1024
  int tws = 1;                   // table stride: w_n^k = tw[k * tws]
  const double2 *tw = nullptr;   // roots e^{-2 pi i k / N}, k < N
  const uint16_t *pos = nullptr; // pos[k]: slot of frequency k after the last stage
  const uint16_t *rev = nullptr; // rev[b]: frequency of the last stage's butterfly b, first output
  const uint16_t *ord = nullptr; // ord[t]: the butterfly b with rev[b] = t
};

__device__ __forceinline__ double2 operator+(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 operator-(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 fft_mul(double2 a, double2 b) {
  return make_double2(__builtin_fma(a.x, b.x, -(a.y * b.y)), __builtin_fma(a.x, b.y, a.y * b.x));
}
// times the root w (DIR < 0) or its conjugate (DIR > 0)
template <int DIR>
__device__ __forceinline__ double2 fft_tw(double2 a, double2 w) {
  if constexpr (DIR > 0) w.y = -w.y;
  return fft_mul(a, w);
}
// times e^{DIR i pi / 2}
template <int DIR>
__device__ __forceinline__ double2 fft_i(double2 a) {
  return DIR < 0 ? make_double2(a.y, -a.x) : make_double2(-a.y, a.x);
}

// x[k] <- sum_n x[n] e^{DIR 2 pi i n k / R}
template <int R, int DIR>
__device__ __forceinline__ void fft_bf(double2 (&x)[R]) {
  if constexpr (R == 2) {
    const double2 a = x[0], b = x[1];
    x[0] = a + b;
    x[1] = a - b;
  } else if constexpr (R == 4) {
    const double2 s02 = x[0] + x[2], d02 = x[0] - x[2], s13 = x[1] + x[3], d13 = fft_i<DIR>(x[1] - x[3]);
    x[0] = s02 + s13;
    x[1] = d02 + d13;
    x[2] = s02 - s13;
    x[3] = d02 - d13;
  } else if constexpr (R == 8) {
    double2 e[4] = {x[0], x[2], x[4], x[6]}, o[4] = {x[1], x[3], x[5], x[7]};
    fft_bf<4, DIR>(e);
    fft_bf<4, DIR>(o);
    constexpr double h = 0.70710678118654752440;
    const double2 i1 = fft_i<DIR>(o[1]), i3 = fft_i<DIR>(o[3]);
    const double2 w1 = make_double2(h * (o[1].x + i1.x), h * (o[1].y + i1.y));
    const double2 w2 = fft_i<DIR>(o[2]);
    const double2 w3 = make_double2(h * (i3.x - o[3].x), h * (i3.y - o[3].y));
    x[0] = e[0] + o[0];
    x[4] = e[0] - o[0];
    x[1] = e[1] + w1;
    x[5] = e[1] - w1;
    x[2] = e[2] + w2;
    x[6] = e[2] - w2;
    x[3] = e[3] + w3;
    x[7] = e[3] - w3;
  } else if constexpr (R == 3) {
    constexpr double s3 = 0.86602540378443864676;
    const double2 s = x[1] + x[2], d = fft_i<DIR>(x[1] - x[2]);
    const double2 c = make_double2(__builtin_fma(-0.5, s.x, x[0].x), __builtin_fma(-0.5, s.y, x[0].y));
    x[0] = x[0] + s;
    x[1] = make_double2(__builtin_fma(s3, d.x, c.x), __builtin_fma(s3, d.y, c.y));
    x[2] = make_double2(__builtin_fma(-s3, d.x, c.x), __builtin_fma(-s3, d.y, c.y));
  } else if constexpr (R == 6) {  // 2 x 3: n = 3 n1 + 2 n2, k = 3 k1 + 4 k2 (mod 6)
    double2 a[3] = {x[0], x[2], x[4]}, b[3] = {x[3], x[5], x[1]};
    fft_bf<3, DIR>(a);
    fft_bf<3, DIR>(b);
    x[0] = a[0] + b[0];
    x[3] = a[0] - b[0];
    x[4] = a[1] + b[1];
    x[1] = a[1] - b[1];
    x[2] = a[2] + b[2];
    x[5] = a[2] - b[2];
  } else {  // 5, 7: sums and differences of the mirrored pairs
    constexpr double C5[2] = {0.30901699437494742410, -0.80901699437494742410};
    constexpr double S5[2] = {0.95105651629515357212, 0.58778525229247312917};
    constexpr double C7[3] = {0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624};
    constexpr double S7[3] = {0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048};
    constexpr int H = (R - 1) / 2;
    double2 s[H], d[H], x0 = x[0], sum = x[0];
#pragma unroll
    for (int i = 0; i < H; ++i) {
      s[i] = x[1 + i] + x[R - 1 - i];
      d[i] = fft_i<DIR>(x[1 + i] - x[R - 1 - i]);
      sum = sum + s[i];
    }
    x[0] = sum;
#pragma unroll
    for (int k = 1; k <= H; ++k) {
      double2 c = x0, t = make_double2(0.0, 0.0);
#pragma unroll
      for (int i = 1; i <= H; ++i) {
        const int m = (k * i) % R;                 // cos even, sin odd about R / 2
        const int f = m <= H ? m : R - m;
        const double cv = R == 5 ? C5[f - 1] : C7[f - 1];
        const double sv = (m <= H ? 1.0 : -1.0) * (R == 5 ? S5[f - 1] : S7[f - 1]);
        c.x = __builtin_fma(cv, s[i - 1].x, c.x);
        c.y = __builtin_fma(cv, s[i - 1].y, c.y);
        t.x = __builtin_fma(sv, d[i - 1].x, t.x);
        t.y = __builtin_fma(sv, d[i - 1].y, t.y);
      }
      x[k] = c + t;
      x[R - k] = c - t;
    }
  }
}

// One stage over the butterflies q, q + dq, ... of a line: ld(slot) and st(slot, t, r, v)
// read and write elements (t, r: butterfly and output, for the last stage's order). LAST:
// no roots. ord: the butterfly to take t-th (a last stage that writes frequencies in
// sequence). The roots are requested with the elements, not once these have arrived.
template <int R, int DIR, bool LAST, class LD, class ST>
__device__ __forceinline__ void fft_stage_r(const FftLen &p, int s, const double2 *tw, int q, int dq, LD ld, ST st,
                                            const uint16_t *ord) {
  const int nb = p.n / R, L = p.len[s], m = LAST ? 1 : L / R, step = (p.n / L) * p.tws;
  for (int t = q; t < nb; t += dq) {
    const int b = ord ? (int)ord[t] : t;
    const int blk = LAST ? b : (int)(((unsigned)b * (unsigned)p.inv[s]) >> 20), j = b - blk * m, base = blk * L + j;
    double2 x[R], w[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      x[r] = ld(base + r * m);
      if constexpr (!LAST)
        if (r > 0) w[r] = tw[j * r * step];
    }
    fft_bf<R, DIR>(x);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if constexpr (!LAST)
        if (r > 0) x[r] = fft_tw<DIR>(x[r], w[r]);
      st(base + r * m, t, r, x[r]);
    }
  }
}
template <int DIR, bool LAST, class LD, class ST>
__device__ __forceinline__ void fft_stage(const FftLen &p, int s, const double2 *tw, int q, int dq, LD ld, ST st,
                                          const uint16_t *ord = nullptr) {
  switch (p.rad[s]) {
    case 2: fft_stage_r<2, DIR, LAST>(p, s, tw, q, dq, ld, st, ord); break;
    case 3: fft_stage_r<3, DIR, LAST>(p, s, tw, q, dq, ld, st, ord); break;
    case 4: fft_stage_r<4, DIR, LAST>(p, s, tw, q, dq, ld, st, ord); break;
    case 5: fft_stage_r<5, DIR, LAST>(p, s, tw, q, dq, ld, st, ord); break;
    case 6: fft_stage_r<6, DIR, LAST>(p, s, tw, q, dq, ld, st, ord); break;
    case 7: fft_stage_r<7, DIR, LAST>(p, s, tw, q, dq, ld, st, ord); break;
    default: fft_stage_r<8, DIR, LAST>(p, s, tw, q, dq, ld, st, ord); break;
  }
}

// A real lattice transform's plan: lengths N (passes along a and b) and N/2 (pass along c)
// over one table of N roots. Owned by a spectrum plan or a Psi grid.
struct FftPlan {
  int64_t N = 0;
  FftLen full, half;
  void *tables = nullptr;

  static bool supports(int64_t N);  // even, at most FFT_MAX_N, no prime factor above 7
  cf_status init(int64_t N);
  void release();
};

// What the first pass of an inverse transform multiplies the half spectrum by, as a
// function of s = |n|^2: nothing, table[s] * mul, or table[s] / div.
struct FftScale {
  const double *table = nullptr;
  double mul = 1.0, div = 0.0;
};

// Passes. `spec` is scratch of N^2 * pitch entries, pitch = fft_pitch(N): the half spectrum
// between passes, its rows padded to whole 128-byte lines (rows of N/2 + 1 entries in
// place of it cost 90 against 52 us a pass at N=256). Spectra outside have rows of
// N/2 + 1 entries, or of `pitch` where they are `spec` itself.
// Forward: real N^3 -> half spectrum `out`. `in` is only read.
cf_status fft_forward(const FftPlan &p, const double *in, double2 *spec, double2 *out, hipStream_t st);
// The same up to the pass along a, which leaves only folded powers: fold[a'][b][c] =
// |f(a', b, c)|^2 + |f(N - a', b, c)|^2 (a' = 0 and N/2 once), (N/2 + 1) * N rows of pitch
// doubles.
cf_status fft_forward_fold(const FftPlan &p, const double *in, double2 *spec, double *fold, hipStream_t st);
// Inverse: half spectrum `in` (unchanged unless it is spec) -> real N^3.
cf_status fft_inverse(const FftPlan &p, const double2 *in, double2 *spec, const FftScale &scale, double *out,
                      hipStream_t st);
// Inverse of two fields from one spectrum R (in fft_line_index's order, `pitch` a multiple of
// eight; only read): R times tab's x and y -> out, out + N^3. tab: a row of `pitch` factors (by c) for
// every pair a' >= b' of folded indices, row a' (a' + 1) / 2 + b' (a table over s = a'^2 +
// b'^2 + c^2 would be an eighth of the size, but every look-up a line of its own: 0.77 ms
// for the first pass at N=384). `spec` is scratch of 2 * N^2 * pitch entries.
cf_status fft_inverse_pair(const FftPlan &p, const double2 *R, const double2 *tab, double2 *spec, int64_t pitch,
                           double *out, hipStream_t st);

// Where fft_inverse_pair's R holds entry (a, b, c): four columns' lines along a lie together,
// so a block of its first pass (four columns, both fields) reads one run of 64 N bytes. In
// rows it read half a 128-byte line per element, each in another plane (N=384 522 against 495 us for the pass).
constexpr int FFT_LW = FFT_CW / 2;
__host__ __device__ __forceinline__ int64_t fft_line_index(int64_t N, int64_t pitch, int64_t a, int64_t b, int64_t c) {
  return ((b * (pitch / FFT_LW) + c / FFT_LW) * N + a) * FFT_LW + c % FFT_LW;
}

// Rows of fft_inverse_pair's table.
inline int64_t fft_pair_rows(int64_t N) { return (N / 2 + 1) * (N / 2 + 2) / 2; }

// Row pitch of internal half spectra: a multiple of eight entries (128 bytes).
inline int64_t fft_pitch(int64_t N) { return (N / 2 + 1 + FFT_CW - 1) / FFT_CW * FFT_CW; }

}  // namespace cf
