// cf_fft.hip -- the passes of the real transforms (cf_fft.hpp) and their plans.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "cf_fft.hpp"

namespace cf {

// Line groups of a pass along a or b: block x -> (c tile, row). Element e of the group's
// line l is at base + row * row_stride + e * e_stride + c0 + l.
struct ColGeom {
  int64_t row_stride, e_stride;  // complex entries
  int nct;                       // c tiles
  int ncol;                      // columns that exist (N/2 + 1, or the pitch when the padding may be touched)
};

// Tables behind the data in LDS: [n][FFT_CW] data, the N roots, one index table. Their
// loads are issued at the kernel's start and their LDS writes done after the first stage,
// which reads its roots from global memory: its own loads then wait for nothing, and the
// barrier after it covers the tables.
struct FftTables {
  const FftLen &p;
  double2 *tw;
  uint16_t *idx;
  const uint16_t *src;
  int n_idx;
  double2 t0, t1;  // this thread's first entries (all of them where 2 threads >= N)
  uint16_t i0;
  __device__ __forceinline__ FftTables(const FftLen &len, double2 *data, const uint16_t *index, int n)
      : p(len), tw(data + (size_t)len.n * FFT_CW), src(index), n_idx(n) {
    const int N = p.n * p.tws, t = (int)threadIdx.x;
    idx = reinterpret_cast<uint16_t *>(tw + N);
    t0 = p.tw[t < N ? t : 0];
    t1 = p.tw[t + (int)blockDim.x < N ? t + (int)blockDim.x : 0];
    i0 = src[t < n_idx ? t : 0];
  }
  __device__ __forceinline__ void store() {
    const int N = p.n * p.tws, t = (int)threadIdx.x, nt = (int)blockDim.x;
    if (t < N) tw[t] = t0;
    if (t + nt < N) tw[t + nt] = t1;
    if (t < n_idx) idx[t] = i0;
    for (int i = t + 2 * nt; i < N; i += nt) tw[i] = p.tw[i];
    for (int i = t + nt; i < n_idx; i += nt) idx[i] = src[i];
  }
};

__device__ __forceinline__ int fft_fold(int i, int N) { return i <= N / 2 ? i : N - i; }

// All stages of the block's lines but the last: gl(e) reads element e of this thread's line
// from global memory, the rest happens in LDS; ends with a barrier.
template <int DIR, class GL>
__device__ __forceinline__ void fft_front(const FftLen &p, double2 *d, FftTables &tb, int q, int dq, GL gl) {
  auto lds_ld = [&](int e) { return d[e * FFT_CW]; };
  auto lds_st = [&](int e, int, int, double2 v) { d[e * FFT_CW] = v; };
  fft_stage<DIR, false>(p, 0, p.tw, q, dq, gl, lds_st);
  tb.store();
  for (int s = 1; s < p.stages - 1; ++s) {
    __syncthreads();
    fft_stage<DIR, false>(p, s, tb.tw, q, dq, lds_ld, lds_st);
  }
  __syncthreads();
}

// Pass along a or b, in place or from `in` to `out`. Contiguous blocks on an XCD: those whose
// rows share 128-byte lines (packed rows of N/2 + 1 entries, the folded powers' half lines)
// meet in one L2. Dealt out in turn, each XCD wrote its part of such a line by itself (pass
// along a into packed rows: N=384 350 -> 264 us, N=512 855 -> 644; folded: 200 -> 179, 416
// -> 373). SCALE: times the scale at s. FOLD:
// powers folded over the pass's axis instead of the spectrum.
template <int DIR, bool SCALE, bool FOLD>
__global__ __launch_bounds__(512) void k_fft_cols(FftLen p, ColGeom gi, ColGeom go, const double2 *in, double2 *out,
                                                  FftScale sc, double *__restrict__ fold) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  double2 *data = reinterpret_cast<double2 *>(smem_raw);
  const int last = p.stages - 1, nbl = p.n / p.rad[last];
  FftTables tb(p, data, FOLD ? p.pos : p.rev, FOLD ? p.n : nbl);
  const int l = threadIdx.x & (FFT_CW - 1), q = threadIdx.x / FFT_CW, dq = blockDim.x / FFT_CW;
  const int block = xcd_order((int)blockIdx.x, (int)gridDim.x), ct = block % gi.nct, row = block / gi.nct;
  const int c = ct * FFT_CW + l;
  const bool rd = c < gi.ncol, wr = c < go.ncol;
  const double2 *src = in + (int64_t)row * gi.row_stride + c;
  double2 *dst = out + (int64_t)row * go.row_stride + c;
  [[maybe_unused]] const int rf = fft_fold(row, p.n), s0 = rf * rf + c * c;
  auto gl = [&](int e) -> double2 {
    if (!rd) return make_double2(0.0, 0.0);
    double2 v = src[(int64_t)e * gi.e_stride];
    if constexpr (SCALE) {
      const int ef = fft_fold(e, p.n), s = s0 + ef * ef;
      const double m = sc.div != 0.0 ? sc.table[s] / sc.div : sc.table[s] * sc.mul;
      v.x *= m;
      v.y *= m;
    }
    return v;
  };
  double2 *d = data + l;
  auto lds_ld = [&](int e) { return d[e * FFT_CW]; };
  if constexpr (FOLD) {
    // powers into the slots of the last stage, then the mirrored pairs
    auto pw = [&](int e, int, int, double2 v) { d[e * FFT_CW].x = v.x * v.x + v.y * v.y; };
    if (last == 0) {
      fft_stage<DIR, true>(p, 0, p.tw, q, dq, gl, pw);
      tb.store();
    } else {
      fft_front<DIR>(p, d, tb, q, dq, gl);
      fft_stage<DIR, true>(p, last, tb.tw, q, dq, lds_ld, pw);
    }
    __syncthreads();
    if (!wr) return;
    double *fr = fold + (int64_t)row * go.row_stride + c;
    for (int k = q; k <= p.n / 2; k += dq) {
      double v = d[tb.idx[k] * FFT_CW].x;
      if (k != 0 && 2 * k != p.n) v += d[tb.idx[p.n - k] * FFT_CW].x;
      fr[(int64_t)k * go.e_stride] = v;
    }
  } else {
    if (last == 0) {  // one butterfly per line: rev[0] = 0
      fft_stage<DIR, true>(p, 0, p.tw, q, dq, gl, [&](int, int, int r, double2 v) {
        if (wr) dst[(int64_t)r * go.e_stride] = v;
      });
      return;
    }
    fft_front<DIR>(p, d, tb, q, dq, gl);
    fft_stage<DIR, true>(p, last, tb.tw, q, dq, lds_ld, [&](int, int t, int r, double2 v) {
      if (wr) dst[(int64_t)((int)tb.idx[t] + r * nbl) * go.e_stride] = v;
    });
  }
}

// Thread roles of the passes along c (cf_fft.hpp): at memory (lm, qm) eight lanes run along
// a row; in between (l, q) they run across the rows.
struct RowRole {
  int l, q, lm, qm, dq;
  // pair: the two lines of a row hold interleaved fields, neighbouring lanes take both
  __device__ __forceinline__ explicit RowRole(bool pair = false) {
    const int t = (int)threadIdx.x;
    l = t & (FFT_CW - 1);
    q = t / FFT_CW;
    lm = pair ? ((t >> 4) & 3) * 2 + (t & 1) : (t >> 3) & 7;
    qm = (pair ? (t >> 1) & 7 : t & 7) | ((t >> 6) << 3);
    dq = (int)blockDim.x / FFT_CW;
  }
};
// LDS slot of element e of line l.
__device__ __forceinline__ int row_slot(const FftLen &p, int e, int l) {
  const int d1 = (int)(((unsigned)e * (unsigned)p.inv[0]) >> 20);
  return e * FFT_CW + ((l + e + d1) & (FFT_CW - 1));
}

// Pass along c of the forward transform: eight rows of N reals -> N/2 + 1 entries. A row is
// taken as N/2 complex numbers z; with Z their transform, X[k] = (Z[k] + conj Z[n-k]) / 2
// - i w^k (Z[k] - conj Z[n-k]) / 2, n = N/2, w = e^{-2 pi i / N}.
__global__ __launch_bounds__(512) void k_fft_r2c(FftLen p, const double2 *__restrict__ in, double2 *__restrict__ out,
                                                 int64_t pitch, int64_t rows) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  double2 *data = reinterpret_cast<double2 *>(smem_raw);
  FftTables tb(p, data, p.pos, p.n);
  const RowRole w;
  const int64_t row = (int64_t)blockIdx.x * FFT_CW + w.lm;
  const bool ok = row < rows;
  const double2 *src = in + (ok ? row : 0) * p.n;
  auto st_m = [&](int e, int, int, double2 v) { data[row_slot(p, e, w.lm)] = v; };
  auto gl = [&](int e) { return src[e]; };
  auto lds_ld = [&](int e) { return data[row_slot(p, e, w.l)]; };
  auto lds_st = [&](int e, int, int, double2 v) { data[row_slot(p, e, w.l)] = v; };
  const int last = p.stages - 1;
  if (last == 0) {
    fft_stage<-1, true>(p, 0, p.tw, w.qm, w.dq, gl, st_m);
    tb.store();
  } else {
    fft_stage<-1, false>(p, 0, p.tw, w.qm, w.dq, gl, st_m);
    tb.store();
    for (int s = 1; s < last; ++s) {
      __syncthreads();
      fft_stage<-1, false>(p, s, tb.tw, w.q, w.dq, lds_ld, lds_st);
    }
    __syncthreads();
    fft_stage<-1, true>(p, last, tb.tw, w.q, w.dq, lds_ld, lds_st);
  }
  __syncthreads();
  if (!ok) return;
  double2 *dst = out + row * pitch;
  const int n = p.n;
  for (int k = w.qm; k <= n / 2; k += w.dq) {
    const double2 z = data[row_slot(p, tb.idx[k], w.lm)];
    if (k == 0) {
      dst[0] = make_double2(z.x + z.y, 0.0);
      dst[n] = make_double2(z.x - z.y, 0.0);
      continue;
    }
    const double2 y = data[row_slot(p, tb.idx[n - k], w.lm)];
    const double2 e = make_double2(0.5 * (z.x + y.x), 0.5 * (z.y - y.y));  // even part
    const double2 o = make_double2(0.5 * (z.y + y.y), 0.5 * (y.x - z.x));  // odd part: -i (Z[k] - conj Z[n-k]) / 2
    const double2 t = fft_mul(o, tb.tw[k]);
    dst[k] = e + t;
    if (2 * k != n) dst[n - k] = make_double2(e.x - t.x, t.y - e.y);
  }
}

// Pass along c of the inverse transform: eight rows of N/2 + 1 entries -> N reals (the
// imaginary parts of the first and last entry are ignored). z[j] = x[2j] + i x[2j+1] is
// the inverse transform of Z[k] = (X[k] + conj X[n-k]) + i w^{-k} (X[k] - conj X[n-k]).
// PAIR: `in` holds two fields interleaved by entry, a block takes four rows of both, and the
// second field goes to out + rows * N/2.
template <bool PAIR>
__global__ __launch_bounds__(512) void k_fft_c2r(FftLen p, const double2 *__restrict__ in, int64_t pitch,
                                                 double2 *__restrict__ out, int64_t rows) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  double2 *data = reinterpret_cast<double2 *>(smem_raw);
  const int last = p.stages - 1, nbl = p.n / p.rad[last];
  FftTables tb(p, data, p.ord, nbl);
  const RowRole w(PAIR);
  constexpr int KS = PAIR ? 2 : 1;  // entry stride
  const int64_t row = PAIR ? (int64_t)blockIdx.x * (FFT_CW / 2) + (w.lm >> 1) : (int64_t)blockIdx.x * FFT_CW + w.lm;
  const int f = PAIR ? w.lm & 1 : 0;
  const bool ok = row < rows;
  const double2 *src = in + (ok ? row : 0) * pitch * KS + f;
  double2 *dst = out + ((ok ? row : 0) + f * rows) * p.n;
  const int n = p.n;
  // Z[k] and Z[n-k] from X[k] and X[n-k], four pairs in flight
  for (int k0 = w.qm; k0 <= n / 2; k0 += 4 * w.dq) {
    double2 a[4], b[4], r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = k0 + i * w.dq <= n / 2 ? k0 + i * w.dq : 0;
      a[i] = src[k * KS];
      b[i] = src[(n - k) * KS];
      r[i] = p.tw[k];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = k0 + i * w.dq;
      if (k > n / 2) break;
      if (k == 0) a[i].y = b[i].y = 0.0;
      const double2 e = make_double2(a[i].x + b[i].x, a[i].y - b[i].y), m = make_double2(a[i].x - b[i].x, a[i].y + b[i].y);
      const double2 t = fft_tw<1>(m, r[i]);  // w^{-k} (X[k] - conj X[n-k])
      data[row_slot(p, k, w.lm)] = make_double2(e.x - t.y, e.y + t.x);
      if (k > 0 && 2 * k != n) data[row_slot(p, n - k, w.lm)] = make_double2(e.x + t.y, t.x - e.y);
    }
  }
  tb.store();
  __syncthreads();
  auto ld_m = [&](int e) { return data[row_slot(p, e, w.lm)]; };
  auto lds_ld = [&](int e) { return data[row_slot(p, e, w.l)]; };
  auto lds_st = [&](int e, int, int, double2 v) { data[row_slot(p, e, w.l)] = v; };
  auto gs = [&](int, int t, int r, double2 v) {  // ord puts frequency t first
    if (ok) dst[t + r * nbl] = v;
  };
  for (int s = 0; s < last; ++s) {
    fft_stage<1, false>(p, s, tb.tw, w.q, w.dq, lds_ld, lds_st);
    __syncthreads();
  }
  fft_stage<1, true>(p, last, tb.tw, w.qm, w.dq, ld_m, gs, tb.idx);
}

// Passes along b and c of the inverse transform of small lattices at once: a block takes a
// plane of N rows through both in LDS (rows of an odd number of entries, so that lanes across
// the rows use different banks). What bounds it is what it saves a launch of: memory latency,
// 3.7-5 us a pass at N=64 whatever it moves. us for an inverse transform, hipFFT (which takes
// two kernels to N=84) / three passes / here: N=32 10.0 / 11.3 / 9.1, 64 11.5 / 13.9 / 11.7, 80 15.8 / 19.4 /
// 16.7, 96 27.5 / 23.5 / 21.1, 128 37.1 / 31.7 / 31.6; Psi and dPsi/dt 64 23.5 / 26.6 / 24.2, 128 73.8 / 67.0 / 59.4.
// PAIR: `in` holds two fields interleaved by entry; a block for each field's planes.
template <bool PAIR>
__global__ __launch_bounds__(512) void k_fft_plane_c2r(FftLen pb, FftLen pc, const double2 *__restrict__ in,
                                                       int64_t pitch, double2 *__restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  const int N = pb.n, n = pc.n, P = (n + 1) | 1, t = (int)threadIdx.x, nt = (int)blockDim.x;
  double2 *data = reinterpret_cast<double2 *>(smem_raw), *tw = data + (size_t)N * P;
  uint16_t *posb = reinterpret_cast<uint16_t *>(tw + N), *posc = posb + N;
  const int a = PAIR ? (int)blockIdx.x >> 1 : (int)blockIdx.x, f = PAIR ? (int)blockIdx.x & 1 : 0;
  constexpr int KS = PAIR ? 2 : 1;  // entry stride
  for (int i = t; i < N; i += nt) {
    tw[i] = pb.tw[i];
    posb[i] = pb.pos[i];
    if (i < n) posc[i] = pc.pos[i];
  }
  const int l = t & (FFT_CW - 1), g = t / FFT_CW, groups = nt / FFT_CW;
  {  // along b: lanes over columns; row slots end in digit-reversed order (posb)
    const int tiles = (n + FFT_CW) / FFT_CW, dq = groups / tiles, q = g / tiles, c = g % tiles * FFT_CW + l;
    const bool on = q < dq && c <= n;
    const double2 *src = in + ((int64_t)a * N * pitch + c) * KS + f;
    double2 *d = data + c;
    auto gl = [&](int e) { return src[e * pitch * KS]; };
    auto ld = [&](int e) { return d[e * P]; };
    auto st = [&](int e, int, int, double2 v) { d[e * P] = v; };
    const int last = pb.stages - 1;
    if (last == 0) {
      if (on) fft_stage<1, true>(pb, 0, pb.tw, q, dq, gl, st);
    } else {
      if (on) fft_stage<1, false>(pb, 0, pb.tw, q, dq, gl, st);
      for (int s = 1; s < last; ++s) {
        __syncthreads();
        if (on) fft_stage<1, false>(pb, s, tw, q, dq, ld, st);
      }
      __syncthreads();
      if (on) fft_stage<1, true>(pb, last, tw, q, dq, ld, st);
    }
  }
  __syncthreads();
  for (int i = t; i < N * (n / 2 + 1); i += nt) {  // Z[k] and Z[n-k] from X[k] and X[n-k] (k_fft_c2r)
    const int k = i / N;
    double2 *d = data + (i - k * N) * P;
    double2 x = d[k], y = d[n - k];
    if (k == 0) x.y = y.y = 0.0;
    const double2 e = make_double2(x.x + y.x, x.y - y.y), m = make_double2(x.x - y.x, x.y + y.y);
    const double2 v = fft_tw<1>(m, tw[k]);
    d[k] = make_double2(e.x - v.y, e.y + v.x);
    if (k > 0 && 2 * k != n) d[n - k] = make_double2(e.x + v.y, v.x - e.y);
  }
  {  // along c: lanes over rows
    const int tiles = (N + FFT_CW - 1) / FFT_CW, dq = groups / tiles, q = g / tiles, r = g % tiles * FFT_CW + l;
    const bool on = q < dq && r < N;
    double2 *d = data + r * P;
    auto ld = [&](int e) { return d[e]; };
    auto st = [&](int e, int, int, double2 v) { d[e] = v; };
    const int last = pc.stages - 1;
    for (int s = 0; s < last; ++s) {
      __syncthreads();
      if (on) fft_stage<1, false>(pc, s, tw, q, dq, ld, st);
    }
    __syncthreads();
    if (on) fft_stage<1, true>(pc, last, tw, q, dq, ld, st);
  }
  __syncthreads();
  double2 *dst = out + ((int64_t)f * N + a) * N * n;
  for (int i = t; i < N * n; i += nt) {
    const int j = i / n;
    dst[i] = data[posb[j] * P + posc[i - j * n]];
  }
}

// First pass (along a) of the inverse of two fields: in * tab.x and in * tab.y into the two
// fields of `out`, interleaved by column ([a][b][c][field]). A block's eight lines are four
// columns of both fields, so the spectrum and the factors are read once and the stores
// still fill whole lines; blocks x and x + 8 (one XCD) share the lines of factors they read.
// (Separate field arrays at N=384: half-line stores 0.53 ms, a block per field 0.68, two
// buffers and one block per CU 0.66; here 0.50.) What bounds it: two blocks a CU, each with
// 24 KB of reads, its stages and 49 KB of stores in sequence. The stores alone take 0.24
// ms, without the factors it is no faster, and a third block (roots read from memory
// instead of LDS, 96 VGPRs) spills: 0.9.
__global__ __launch_bounds__(512) void k_fft_pair(FftLen p, const double2 *__restrict__ in,
                                                  const double2 *__restrict__ tab, double2 *__restrict__ out,
                                                  int pitch) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  double2 *data = reinterpret_cast<double2 *>(smem_raw);
  const int last = p.stages - 1, nbl = p.n / p.rad[last];
  FftTables tb(p, data, p.rev, nbl);
  const int l = threadIdx.x & (FFT_CW - 1), q = threadIdx.x / FFT_CW, dq = blockDim.x / FFT_CW;
  const int nct = pitch / FFT_CW, tile = (int)((blockIdx.x >> 4) << 3) + (int)(blockIdx.x & 7);
  const int ct = 2 * (tile % nct) + ((int)(blockIdx.x >> 3) & 1), row = tile / nct, f = l & 1;
  if (row >= p.n) return;  // the grid is rounded up to pairs of eight blocks
  const int c = ct * (FFT_CW / 2) + (l >> 1);
  const bool rd = c <= p.n / 2;
  const int64_t e_stride = (int64_t)p.n * pitch;
  const double2 *src = in + fft_line_index(p.n, pitch, 0, row, c);
  double2 *dst = out + 2 * ((int64_t)row * pitch + c) + f;
  const int rf = fft_fold(row, p.n);
  auto gl = [&](int e) -> double2 {
    if (!rd) return make_double2(0.0, 0.0);
    const int ef = fft_fold(e, p.n), hi = ef > rf ? ef : rf, lo = ef > rf ? rf : ef;
    const double2 x = src[e * FFT_LW], t = tab[(int64_t)(hi * (hi + 1) / 2 + lo) * pitch + c];
    const double m = f == 0 ? t.x : t.y;
    return make_double2(x.x * m, x.y * m);
  };
  double2 *d = data + l;
  if (last == 0) {
    fft_stage<1, true>(p, 0, p.tw, q, dq, gl, [&](int, int, int r, double2 v) { dst[2 * r * e_stride] = v; });
    return;
  }
  fft_front<1>(p, d, tb, q, dq, gl);
  fft_stage<1, true>(p, last, tb.tw, q, dq, [&](int e) { return d[e * FFT_CW]; }, [&](int, int t, int r, double2 v) {
    dst[2 * ((int)tb.idx[t] + r * nbl) * e_stride] = v;
  });
}

// ---------------------------------------------------------------- plans
bool FftPlan::supports(int64_t N) {
  if (N < 4 || N % 2 || N > FFT_MAX_N) return false;
  for (int f : {2, 3, 5, 7})
    while (N % f == 0) N /= f;
  return N == 1;
}

// Radices of n, the widest first: eights, then fours, a two merged with a three into a six.
static std::vector<int> fft_radices(int n) {
  int e2 = 0, e3 = 0;
  std::vector<int> r, tail;
  while (n % 7 == 0) { tail.push_back(7); n /= 7; }
  while (n % 5 == 0) { tail.push_back(5); n /= 5; }
  while (n % 3 == 0) { ++e3; n /= 3; }
  while (n % 2 == 0) { ++e2; n /= 2; }
  if (e2 % 3 == 1 && e3 > 0) {  // 2 * 3
    --e2;
    --e3;
    tail.push_back(6);
  }
  while (e2 >= 3 && e2 != 4) { r.push_back(8); e2 -= 3; }
  while (e2 >= 2) { r.push_back(4); e2 -= 2; }
  r.insert(r.end(), tail.begin(), tail.end());
  r.insert(r.end(), (size_t)e3, 3);
  r.insert(r.end(), (size_t)e2, 2);
  if (r.empty()) r.push_back(1);
  return r;
}

static bool fft_len(int n, int tws, FftLen *p, std::vector<uint16_t> *pos, std::vector<uint16_t> *rev,
                    std::vector<uint16_t> *ord) {
  const std::vector<int> rad = fft_radices(n);
  if (rad.size() > FFT_MAX_STAGES || rad[0] < 2) return false;
  p->n = n;
  p->tws = tws;
  p->stages = (int)rad.size();
  int L = n;
  for (size_t s = 0; s < rad.size(); ++s) {
    p->rad[s] = rad[s];
    p->len[s] = L;
    const int m = L / rad[s];
    p->inv[s] = ((1 << 20) + m - 1) / m;
    for (int b = 0; b < (s == 0 ? n : n / rad[s]); ++b)  // (row_slot divides elements by the first stride)
      if ((int)(((unsigned)b * (unsigned)p->inv[s]) >> 20) != b / m) return false;
    L = m;
  }
  // slot = d1 (n/R1) + d2 (n/(R1 R2)) + ..., frequency = d1 + R1 d2 + R1 R2 d3 + ...
  pos->assign((size_t)n, 0);
  const int last = rad.back();
  rev->assign((size_t)(n / last), 0);
  for (int slot = 0; slot < n; ++slot) {
    int rest = slot, span = n, k = 0, scale = 1;
    for (int R : rad) {
      span /= R;
      k += (rest / span) * scale;
      rest %= span;
      scale *= R;
    }
    (*pos)[(size_t)k] = (uint16_t)slot;
    if (slot % last == 0) (*rev)[(size_t)(slot / last)] = (uint16_t)k;
  }
  ord->assign(rev->size(), 0);
  for (size_t b = 0; b < rev->size(); ++b) (*ord)[(*rev)[b]] = (uint16_t)b;
  return true;
}

// Dynamic LDS above 64 KB (N > 448) has to be asked for, per kernel and device.
static cf_status fft_allow_lds() {
  constexpr int most = 160 << 10;
  const void *kernels[] = {(const void *)k_fft_r2c,  (const void *)k_fft_c2r<false>, (const void *)k_fft_c2r<true>,
                           (const void *)k_fft_plane_c2r<false>, (const void *)k_fft_plane_c2r<true>,
                           (const void *)k_fft_pair, (const void *)k_fft_cols<-1, false, false>,
                           (const void *)k_fft_cols<-1, false, true>, (const void *)k_fft_cols<1, false, false>,
                           (const void *)k_fft_cols<1, true, false>};
  for (const void *k : kernels) CF_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, most));
  return CF_OK;
}

cf_status FftPlan::init(int64_t n_sites) {
  CF_REQUIRE(supports(n_sites), "transform size N=%lld has a prime factor above 7 or exceeds %d", (long long)n_sites,
             FFT_MAX_N);
  CF_TRY(fft_allow_lds());
  N = n_sites;
  const int n = (int)N;
  std::vector<uint16_t> posf, revf, ordf, posh, revh, ordh;
  CF_REQUIRE(fft_len(n, 1, &full, &posf, &revf, &ordf) && fft_len(n / 2, 2, &half, &posh, &revh, &ordh),
             "transform size N=%lld: no stage plan", (long long)N);
  std::vector<double2> tw((size_t)n);
  for (int k = 0; k < n; ++k) {
    // octant reduction: sines and cosines of at most pi/4, in extended precision
    const long double pi = 3.14159265358979323846264338327950288L;
    const int e = 8 * k;  // angle = 2 pi k / n; octant index and its remainder
    const int oct = e / n;
    const long double a = 2.0L * pi * (long double)k / (long double)n;
    long double c, s;
    switch (oct) {
      case 0: c = cosl(a); s = sinl(a); break;
      case 1: case 2: { const long double b = 2.0L * pi * (long double)(4 * k - n) / (4.0L * n); c = -sinl(b); s = cosl(b); break; }
      case 3: case 4: { const long double b = 2.0L * pi * (long double)(2 * k - n) / (2.0L * n); c = -cosl(b); s = -sinl(b); break; }
      case 5: case 6: { const long double b = 2.0L * pi * (long double)(4 * k - 3 * n) / (4.0L * n); c = sinl(b); s = -cosl(b); break; }
      default: { const long double b = 2.0L * pi * (long double)(k - n) / (long double)n; c = cosl(b); s = sinl(b); break; }
    }
    tw[(size_t)k] = make_double2((double)c, (double)-s);
  }
  const size_t bt = tw.size() * sizeof(double2), b16 = sizeof(uint16_t);
  const size_t total = bt + (posf.size() + 2 * revf.size() + posh.size() + 2 * revh.size()) * b16;
  if (hipMalloc(&tables, total) != hipSuccess) {
    set_error("transform plan N=%lld: device allocation failed", (long long)N);
    tables = nullptr;
    return CF_E_NOMEM;
  }
  std::vector<char> host(total);
  size_t at = 0;
  auto put = [&](const void *src, size_t bytes) {
    memcpy(host.data() + at, src, bytes);
    at += bytes;
    return (const void *)((const char *)tables + (at - bytes));
  };
  full.tw = half.tw = (const double2 *)put(tw.data(), bt);
  full.pos = (const uint16_t *)put(posf.data(), posf.size() * b16);
  full.rev = (const uint16_t *)put(revf.data(), revf.size() * b16);
  full.ord = (const uint16_t *)put(ordf.data(), ordf.size() * b16);
  half.ord = (const uint16_t *)put(ordh.data(), ordh.size() * b16);
  half.pos = (const uint16_t *)put(posh.data(), posh.size() * b16);
  half.rev = (const uint16_t *)put(revh.data(), revh.size() * b16);
  if (hipMemcpy(tables, host.data(), total, hipMemcpyHostToDevice) != hipSuccess) {
    set_error("transform plan N=%lld: table upload failed", (long long)N);
    release();
    return CF_E_HIP;
  }
  return CF_OK;
}

void FftPlan::release() {
  if (tables) (void)hipFree(tables);
  tables = nullptr;
  N = 0;
}

static size_t fft_lds(const FftLen &p) {
  return ((size_t)p.n * FFT_CW + (size_t)p.n * p.tws) * sizeof(double2) + (size_t)p.n * sizeof(uint16_t);
}
// Threads per block: LDS bounds the blocks of a CU, together they should be 16 wavefronts.
static unsigned fft_threads(size_t lds) {
  const int blocks = (int)std::max<size_t>(1, (160 << 10) / lds), waves = (16 + blocks - 1) / blocks;
  return 64u * (unsigned)std::min(8, waves);
}

static cf_status pass_r2c(const FftPlan &p, const double *in, double2 *out, int64_t pitch, int64_t rows,
                          hipStream_t st) {
  hipLaunchKernelGGL(k_fft_r2c, dim3((unsigned)cdiv(rows, FFT_CW)), dim3(fft_threads(fft_lds(p.half))), fft_lds(p.half), st,
                     p.half, (const double2 *)in, out, pitch, rows);
  CF_LAUNCHED();
  return CF_OK;
}
template <bool PAIR>
static cf_status pass_c2r(const FftPlan &p, const double2 *in, int64_t pitch, double *out, int64_t rows,
                          hipStream_t st) {
  hipLaunchKernelGGL(k_fft_c2r<PAIR>, dim3((unsigned)cdiv(rows, PAIR ? FFT_CW / 2 : FFT_CW)),
                     dim3(fft_threads(fft_lds(p.half))), fft_lds(p.half), st, p.half, in, pitch, (double2 *)out, rows);
  CF_LAUNCHED();
  return CF_OK;
}

// Largest lattice whose inverse takes the passes along b and c in one kernel. There its plane
// fills a CU's LDS (135 of 160 KB), and one field's inverse is no faster than by two passes
// (above); two fields' still is.
constexpr int FFT_PLANE_N = 128;
template <bool PAIR>
static cf_status pass_plane(const FftPlan &p, const double2 *in, int64_t pitch, double *out, hipStream_t st) {
  const size_t lds = (size_t)p.N * ((p.N / 2 + 1) | 1) * sizeof(double2) + (size_t)p.N * sizeof(double2) +
                     (size_t)(p.N + p.N / 2) * sizeof(uint16_t);
  hipLaunchKernelGGL(k_fft_plane_c2r<PAIR>, dim3((unsigned)(PAIR ? 2 * p.N : p.N)), dim3(512), lds, st, p.full, p.half,
                     in, pitch, (double2 *)out);
  CF_LAUNCHED();
  return CF_OK;
}

// Rows of a pass along b: planes a; along a: rows b.
static ColGeom cols_geom(const FftPlan &p, bool along_a, int64_t pitch) {
  const int64_t H = p.N / 2 + 1, plane = p.N * pitch;
  ColGeom g{along_a ? pitch : plane, along_a ? plane : pitch, (int)cdiv(H, FFT_CW), 0};
  g.ncol = (int)(pitch % FFT_CW == 0 ? pitch : H);
  return g;
}
template <int DIR, bool SCALE, bool FOLD>
static cf_status pass_cols(const FftPlan &p, const ColGeom &gi, const ColGeom &go, int64_t rows, const double2 *in,
                           double2 *out, const FftScale &sc, double *fold, hipStream_t st) {
  const FftLen &l = p.full;
  hipLaunchKernelGGL((k_fft_cols<DIR, SCALE, FOLD>), dim3((unsigned)(gi.nct * rows)), dim3(fft_threads(fft_lds(l))),
                     fft_lds(l), st, l, gi, go, in, out, sc, fold);
  CF_LAUNCHED();
  return CF_OK;
}

cf_status fft_forward(const FftPlan &p, const double *in, double2 *spec, double2 *out, hipStream_t st) {
  const int64_t pitch = fft_pitch(p.N);
  const ColGeom b = cols_geom(p, false, pitch), a = cols_geom(p, true, pitch);
  CF_TRY(pass_r2c(p, in, spec, pitch, p.N * p.N, st));
  CF_TRY((pass_cols<-1, false, false>(p, b, b, p.N, spec, spec, FftScale{}, nullptr, st)));
  return pass_cols<-1, false, false>(p, a, out == spec ? a : cols_geom(p, true, p.N / 2 + 1), p.N, spec, out,
                                     FftScale{}, nullptr, st);
}

cf_status fft_forward_fold(const FftPlan &p, const double *in, double2 *spec, double *fold, hipStream_t st) {
  const int64_t pitch = fft_pitch(p.N);
  const ColGeom b = cols_geom(p, false, pitch), a = cols_geom(p, true, pitch);
  ColGeom f = a;  // the same row and element strides, of doubles
  f.ncol = (int)(p.N / 2 + 1);
  CF_TRY(pass_r2c(p, in, spec, pitch, p.N * p.N, st));
  CF_TRY((pass_cols<-1, false, false>(p, b, b, p.N, spec, spec, FftScale{}, nullptr, st)));
  return pass_cols<-1, false, true>(p, a, f, p.N, spec, spec, FftScale{}, fold, st);
}

cf_status fft_inverse(const FftPlan &p, const double2 *in, double2 *spec, const FftScale &scale, double *out,
                      hipStream_t st) {
  const int64_t pitch = fft_pitch(p.N);
  const ColGeom b = cols_geom(p, false, pitch), a = cols_geom(p, true, pitch);
  ColGeom r = in == spec ? a : cols_geom(p, true, p.N / 2 + 1);
  r.ncol = (int)(p.N / 2 + 1);  // a scale's table ends there
  if (scale.table) CF_TRY((pass_cols<1, true, false>(p, r, a, p.N, in, spec, scale, nullptr, st)));
  else CF_TRY((pass_cols<1, false, false>(p, r, a, p.N, in, spec, scale, nullptr, st)));
  if (p.N <= FFT_PLANE_N) return pass_plane<false>(p, spec, pitch, out, st);
  CF_TRY((pass_cols<1, false, false>(p, b, b, p.N, spec, spec, FftScale{}, nullptr, st)));
  return pass_c2r<false>(p, spec, pitch, out, p.N * p.N, st);
}

cf_status fft_inverse_pair(const FftPlan &p, const double2 *R, const double2 *tab, double2 *spec, int64_t pitch,
                           double *out, hipStream_t st) {
  const int64_t tiles = p.N * (pitch / FFT_CW);
  hipLaunchKernelGGL(k_fft_pair, dim3((unsigned)(cdiv(tiles, 8) * 16)), dim3(fft_threads(fft_lds(p.full))),
                     fft_lds(p.full), st, p.full, R, tab, spec, (int)pitch);
  CF_LAUNCHED();
  if (p.N <= FFT_PLANE_N) return pass_plane<true>(p, spec, pitch, out, st);
  ColGeom b = cols_geom(p, false, 2 * pitch);
  b.nct = (int)(2 * pitch / FFT_CW);
  CF_TRY((pass_cols<1, false, false>(p, b, b, p.N, spec, spec, FftScale{}, nullptr, st)));
  return pass_c2r<true>(p, spec, pitch, out, p.N * p.N, st);
}

}  // namespace cf
