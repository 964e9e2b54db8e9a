// cf_rk4_tb.hip -- temporally blocked classic RK4 on one lattice: all four
// stages of a step in one kernel, so the state is read once and written once
// per step (the step body, its geometry and its arithmetic are described in
// cf_tb_body.hpp). One block per work unit (output tile x a-chunk).
//
// HBM per site-step: FP64 read x, write x' = 32 B; FP32-comp read hi, lo, write
// hi', lo' = 32 B (plus halo and warm-up re-reads, mostly served by L2).
// The output goes to a second buffer (neighbouring blocks still read the old
// state), so runs ping-pong between two state arrays.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <map>
#include <mutex>
#include <tuple>
#include <utility>
#include <vector>

#include "cf_tb_body.hpp"
#include "cf_tb_run.hpp"

namespace cf {

struct TbGeom {
  int64_t N;
  int shape;           // index of the kernel's region shape (below)
  int rb, rc;          // its rows and columns
  int Tb, Tc;          // output tile edges along b and c
  int ntb, ntc;        // tiles along b and c
  int A;               // planes per chunk
  int n_ac;            // chunks
  int total;           // ntb * ntc * n_ac
  int64_t NA;          // planes of the state buffers along a (N, or a slab's planes + ghosts)
  int64_t a_lo, a_hi;  // output planes [a_lo, a_hi)
  int pace;            // ticks of the 100 MHz real-time counter per plane iteration, 0: unpaced
};

// Work unit of logical block `bid`: tile (tb, tc), chunk ac, c fastest.
__device__ __forceinline__ TbUnit tb_unit_of(const TbGeom &g, int bid) {
  const int tc = bid % g.ntc;
  const int rest = bid / g.ntc;
  const int tb = rest % g.ntb;
  const int ac = rest / g.ntb;
  TbUnit u;
  u.N = g.N;
  u.T = g.Tb;
  u.Tc = g.Tc;
  u.b0 = (int64_t)tb * g.Tb;
  u.c0 = (int64_t)tc * g.Tc;
  u.a0 = g.a_lo + (int64_t)ac * g.A;
  u.a1 = (u.a0 + g.A < g.a_hi) ? u.a0 + g.A : g.a_hi;
  u.NA = g.NA;
  u.pace = g.pace;
  return u;
}

// One kernel per storage form, region shape and lambda = 0 / != 0. WAVES: wavefronts
// per SIMD the registers leave room for (512 / WAVES VGPRs each). PACE: the blocks keep
// to a common schedule of plane iterations (cf_tb_body.hpp).
template <int MODE, bool LAM, class SH, int WAVES, bool PACE>
__global__ __launch_bounds__(SH::NT) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES))) void k_rk4_tb(
    TbGeom g, TbStep k, TbStepF kf, const void *xin, const float *lin, void *xout, float *lout) {
  __shared__ __attribute__((aligned(16))) TbElem<MODE, SH> smem[SH::LDS];
  // Blocks go to the 8 XCDs round robin; consecutive logical tiles are mapped
  // to one XCD so that neighbouring tiles' halos meet in its L2.
  tb_unit<MODE, LAM, SH, TB_KG, PACE>(smem, tb_unit_of(g, xcd_order(blockIdx.x, g.total)), k, kf, xin, lin, xout,
                                      lout);
}

// The same step for the equation variants, FP64.
template <int VAR, class SH, int WAVES>
__global__ __launch_bounds__(SH::NT) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES))) void k_rk4_tb_var(
    TbGeom g, TbStep k, const double *xin, double *xout, const double *psi, TbPsi cps) {
  __shared__ __attribute__((aligned(16))) double smem[SH::LDS];
  tb_unit<TB_F64, false, SH, VAR>(smem, tb_unit_of(g, xcd_order(blockIdx.x, g.total)), k, TbStepF{}, xin, nullptr,
                                  xout, nullptr, psi, cps);
}

// Region shapes of the single-lattice kernels, smallest first. A large region repeats
// less of its neighbours' work and reads (26 x 64 tiles: 1.23 region sites per output
// site, 8 x 16 ones 1.88); a small one gives a small lattice enough blocks and takes
// less time per plane.
//
// t1 and tau are the time of a plane iteration in us with one block on a CU and, per
// block, with `resident` blocks, the CU full (states in cache); bw the rate in bytes per us
// at which launches that stream through HBM pass their loads (halo and warm-up included)
// and stores. Measured over N = 32 .. 512 on 256 CUs; see tb_cost.
struct TbShapeInfo {
  int rb, rc, resident;
  double t1, tau, bw;
};
typedef TbShape<12, 20, 2, 128> TbS12x20;
typedef TbShape<14, 36, 2, 256> TbS14x36;
typedef TbShape<28, 36, 2, 512> TbS28x36;
typedef TbShape<30, 68, 2, 1024> TbS30x68;
typedef TbShape<15, 132, 2, 1024> TbS15x132;  // floats: 128-column rows, four lines
typedef TbShape<14, 36, 1, 512> TbC14x36;     // a column per thread (TB_F32C, variants)
typedef TbShape<28, 36, 1, 1024> TbC28x36;
typedef TbShape<22, 68, 2, 768> TbC22x68;     // 768 threads: 168 VGPRs for float histories and double sums

enum : int { TB_FAM_F64 = 0, TB_FAM_F32C = 1, TB_FAM_F32S = 2, TB_FAM_CURV = 3, TB_FAM_SQRT = 4, TB_FAM_COM = 5,
             TB_FAM_APX = 6 };

// Bytes a launch loads per region site and plane iteration: the state, and Psi (fixed
// curvature) or Psi and dPsi/dt at three stage times (comoving; the coarse grid's 1/8).
static const double tb_load_bytes[7] = {16.0, 16.0, 16.0, 24.0, 16.0, 64.0, 22.0};

static const std::vector<TbShapeInfo> &tb_shapes(int family) {
  static const std::vector<TbShapeInfo> t[7] = {
      {{12, 20, 8, 0.68, 0.26, 4.9e6}, {14, 36, 4, 0.70, 0.47, 5.0e6}, {28, 36, 2, 1.00, 0.92, 5.3e6},
       {30, 68, 1, 2.00, 2.00, 5.57e6}},
      {{14, 36, 2, 0.75, 0.58, 4.6e6}, {28, 36, 1, 1.22, 1.22, 4.35e6}, {22, 68, 1, 1.73, 1.73, 5.1e6}},
      {{12, 20, 8, 0.60, 0.18, 3.9e6}, {14, 36, 4, 0.65, 0.39, 4.7e6}, {28, 36, 2, 0.84, 0.78, 4.7e6},
       {30, 68, 1, 1.65, 1.65, 5.15e6}, {15, 132, 1, 1.50, 1.50, 5.85e6}},
      {{14, 36, 2, 0.82, 0.68, 5.3e6}, {28, 36, 1, 1.44, 1.44, 5.1e6}, {22, 68, 1, 1.99, 1.99, 5.5e6}},
      {{14, 36, 2, 1.22, 1.13, 5.0e6}, {28, 36, 1, 2.29, 2.29, 5.0e6}, {22, 68, 1, 3.40, 3.40, 5.2e6}},
      {{14, 36, 2, 1.25, 1.09, 6.1e6}, {28, 36, 1, 2.20, 2.20, 6.0e6}},
      {{14, 36, 2, 1.05, 0.85, 4.0e6}, {28, 36, 1, 1.70, 1.70, 3.85e6}},
  };
  return t[family];
}

// Compute units of the current device.
static int tb_cus() {
  static std::atomic<int> known[64] = {};
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if ((cus = known[dev].load(std::memory_order_relaxed)) > 0) return cus;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) return 256;
  known[dev].store(cus, std::memory_order_relaxed);
  return cus;
}

// Tiles of (rb - 4) x (rc - 4) sites (the whole extent when N is smaller) over the
// output planes [a_lo, a_hi) of buffers of NA planes; a periodic lattice: 0, N, N.
static TbGeom tb_geom(int family, int shape, int64_t N, int A, int64_t a_lo, int64_t a_hi, int64_t NA) {
  const TbShapeInfo &s = tb_shapes(family)[(size_t)shape];
  TbGeom g;
  g.N = N;
  g.shape = shape;
  g.rb = s.rb;
  g.rc = s.rc;
  g.a_lo = a_lo;
  g.a_hi = a_hi;
  g.NA = NA;
  const int64_t planes = a_hi - a_lo;
  g.Tb = N < s.rb - 2 * TBH ? (int)N : s.rb - 2 * TBH;
  g.Tc = N < s.rc - 2 * TBH ? (int)N : s.rc - 2 * TBH;
  g.ntb = (int)cdiv(N, g.Tb);
  g.ntc = (int)cdiv(N, g.Tc);
  g.A = (A <= 0 || A > planes) ? (int)planes : A;
  g.n_ac = (int)cdiv(planes, g.A);
  g.total = g.ntb * g.ntc * g.n_ac;
  g.pace = 0;
  return g;
}

// Modelled time of a launch in us. Few chunks leave CUs idle, many repeat warm-up planes;
// small regions repeat halos. A block takes A + 4 iterations, of which the two that only
// load and the two without k3 and k4 cost two.
//   While all of it fits the 256 MB cache: the larger of the busiest CU's iterations (its n
//   = ceil(blocks / CUs) blocks, `resident` at a time) and the bytes passed at 1.6 bw.
//   Beyond: rounds of CUs * resident blocks, each the larger of its iterations, at 0.7 of
//   the above (what is left of them when the blocks of a round run against each other and
//   HBM), and its bytes at bw; a last round that fills a part of the chip lies by that part
//   between the two. (With the launch's bytes over bw instead, launches a little over a
//   whole number of rounds were picked: N=300, FP64, 420 blocks 212 us, 240 blocks 188.)
// Of the (shape, chunk) pairs measured at 17 sizes, N = 32 .. 512, and every storage form
// and variant, 6 to 30 each, it picks one within 0.4% of the fastest on average, 8% at worst.
static double tb_cost(int family, const TbShapeInfo &s, const TbGeom &g, int cus) {
  const double lb = tb_load_bytes[family], launch = 1.8, it = (double)(g.A + 2);
  const double sites = (double)g.N * (double)g.N * (double)(g.a_hi - g.a_lo);
  const double loads = lb * (double)g.ntb * g.ntc * g.n_ac * s.rb * s.rc * (double)(g.A + 2 * TBH);
  const double bytes = loads + 16.0 * sites;
  if ((lb + 16.0) * sites <= 256e6) {
    const int64_t n = cdiv(g.total, cus), full = n / s.resident, rest = n % s.resident;
    const double last = rest ? std::max(s.t1, (double)rest * s.tau) : 0.0;
    return std::max(launch + it * ((double)full * s.resident * s.tau + last), bytes / (1.6 * s.bw));
  }
  const int64_t slots = (int64_t)cus * s.resident, full = g.total / slots, rest = g.total % slots;
  const double round = std::max(0.7 * s.resident * s.tau * it, bytes / g.total * (double)slots / s.bw);
  double t = launch + (double)full * round;
  if (rest) {
    const double least = 0.7 * std::max(s.t1, (double)cdiv(rest, cus) * s.tau) * it;
    t += least + std::max(round - least, 0.0) * (double)rest / (double)slots;
  }
  return t;
}

// A chunk that the caller gives can leave CUs idle. Beyond the cache their share of the rate
// is lost, so such a launch takes shorter tiles, as many as there are CUs (in doubles four
// fifths of them: beyond that the blocks run against each other). us a step, tiles as large as
// the region / here:
//   float forces, N=256, chunk 128 (24 rows / 16) 179 / 136, 224 of 112 137 / 114, 300 of 300
//     376 / 280, 320 of 320 390 / 310, 512 of 512 1070 / 939
//   FP64: 224 of 112 127 / 113, 250 of 125 138 / 130 (256 blocks: 142), 320 of 320 350 / 310
// FP32-comp and the variants are bound by arithmetic in their largest regions, where shorter
// tiles lose (FP32-comp, N=320, chunk 160 288 / 308): they keep theirs.
static void tb_fill(int family, TbGeom &g) {
  if (family != TB_FAM_F64 && family != TB_FAM_F32S) return;
  const double sites = (double)g.N * (double)g.N * (double)(g.a_hi - g.a_lo);
  if ((tb_load_bytes[family] + 16.0) * sites <= 256e6) return;
  const int cus = tb_cus(), most = family == TB_FAM_F32S ? cus : cus * 4 / 5;
  const int rows = most / (g.ntc * g.n_ac);  // tiles along b that keep to `most` blocks
  if (rows <= g.ntb) return;
  g.Tb = (int)cdiv(g.N, rows);
  g.ntb = (int)cdiv(g.N, g.Tb);
  g.total = g.ntb * g.ntc * g.n_ac;
}

// The cheapest (shape, chunk) of a launch, or the cheapest shape for a given chunk. With
// `near`, also every chunk length whose best shape costs at most near_pct percent more,
// cheapest first. Chunk lengths are the ceil(planes / k); there are about 2 sqrt(planes).
// Measured on MI355X (us a step, FP64; before: one rule over 32 x 32 regions with a halo
// of four): N=32 20.5 -> 3.5, 64 20.7 -> 6.0, 128 31.6 -> 17.8, 200 80 -> 55, 250 152 ->
// 110, 300 258 -> 189, 384 467 -> 392, 512 1239 -> 886.
static TbGeom tb_plan_search(int family, int64_t N, int chunk, int64_t a_lo, int64_t a_hi, int64_t NA,
                             std::vector<int> *near = nullptr, int near_pct = 0) {
  const std::vector<TbShapeInfo> &shapes = tb_shapes(family);
  const int cus = tb_cus();
  const int64_t planes = a_hi - a_lo;
  TbGeom best{};
  double best_cost = -1.0;
  std::vector<std::pair<double, int>> costs;
  auto try_chunk = [&](int A) {
    double least = -1.0;
    for (size_t i = 0; i < shapes.size(); ++i) {
      const TbGeom g = tb_geom(family, (int)i, N, A, a_lo, a_hi, NA);
      const double c = tb_cost(family, shapes[i], g, cus);
      if (least < 0.0 || c < least) least = c;
      if (best_cost < 0.0 || c < best_cost) {
        best = g;
        best_cost = c;
      }
    }
    if (near) costs.emplace_back(least, A);
  };
  if (chunk > 0) {
    try_chunk(chunk);
    tb_fill(family, best);
    return best;
  }
  for (int64_t k = 1; k <= planes;) {  // every distinct ceil(planes / k)
    const int64_t A = cdiv(planes, k);
    try_chunk((int)A);
    k = A > 1 ? (planes + A - 2) / (A - 1) : planes + 1;  // the first k of a shorter chunk
  }
  if (near) {
    std::sort(costs.begin(), costs.end());
    for (const auto &c : costs)
      if (c.first * 100.0 <= best_cost * (100 + near_pct)) near->push_back(c.second);
  }
  return best;
}

// The same, with each thread's last plan of a family kept: a run asks for one geometry step
// after step, and the search over a hundred (shape, chunk) pairs was 0.8 of the 4.1 us of
// host time that a step's call takes at N=128 (0.4 of 4.3 at N=32).
static TbGeom tb_plan(int family, int64_t N, int chunk, int64_t a_lo, int64_t a_hi, int64_t NA) {
  struct Last {
    std::tuple<int64_t, int, int64_t, int64_t, int64_t, int> key{0, 0, 0, 0, 0, 0};  // N = 0: none
    TbGeom g{};
  };
  static thread_local Last last[7];
  const auto key = std::make_tuple(N, chunk, a_lo, a_hi, NA, tb_cus());
  Last &l = last[family];
  if (l.key != key) {
    l.g = tb_plan_search(family, N, chunk, a_lo, a_hi, NA);
    l.key = key;
  }
  return l.g;
}

// Where the FP32-comp run puts its second hi and lo arrays in the work buffer: at the
// first address from `from` on with the same residue modulo TB_ALIGN_SLACK as the
// caller's array `like`, so that each array's offset to its partner of the other step is
// a multiple of 4 KB (offsets that are not cost up to 20%; the work buffer carries the
// slack, cf_rk4_tb_work_bytes).
constexpr size_t TB_ALIGN_SLACK = 4096;
static float *same_residue(void *from, const float *like) {
  const uintptr_t f = reinterpret_cast<uintptr_t>(from), l = reinterpret_cast<uintptr_t>(like);
  return reinterpret_cast<float *>(f + ((l - f) & (TB_ALIGN_SLACK - 1)));
}

// Default chunk of the single-precision-stencil step per device and lattice size, set by
// cf_rk4_tb_tune_pace (chunk <= 0) or cf_rk4_tb_set_chunk; absent: the cost model's.
static std::mutex g_chunk_mu;
static std::map<std::pair<int, int64_t>, int> g_chunk;

static int tb_f32s_tuned_chunk(int64_t N) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  std::lock_guard<std::mutex> lock(g_chunk_mu);
  const auto it = g_chunk.find(std::make_pair(dev, N));
  return it == g_chunk.end() ? 0 : it->second;
}

static TbGeom tb_f64_geom(int64_t N, int chunk) { return tb_plan(TB_FAM_F64, N, chunk, 0, N, N); }

// ... of the single-precision-stencil kernel (sa) or the FP32-comp one.
static TbGeom tb_comp_geom(bool sa, int64_t N, int chunk) {
  if (!sa) return tb_plan(TB_FAM_F32C, N, chunk, 0, N, N);
  if (chunk <= 0) chunk = tb_f32s_tuned_chunk(N);
  return tb_plan(TB_FAM_F32S, N, chunk, 0, N, N);
}

// The regions that cf_rk4_tb_f32s_region reports: those of the step while its regions had
// halos of four, 24 x 40 unless rounds x (chunk + 8) of a launch over 32 x 32 ones was more
// than 20% lower. Kept for callers that hold its answers; what a launch runs over is tb_plan's
// choice (cf_rk4_tb_geometry).
static void tb_f32s_class(int64_t N, int *rows, int *cols) {
  const int cus = tb_cus();
  auto least = [&](int64_t tb, int64_t tc) {
    const int64_t tiles = cdiv(N, N < tb ? N : tb) * cdiv(N, N < tc ? N : tc);
    int64_t best = -1;
    for (int64_t k = 1; k <= (N / 8 > 1 ? N / 8 : 1); ++k) {
      const int64_t ch = cdiv(N, k), c = cdiv(tiles * cdiv(N, ch), cus) * (ch + 8);
      if (cdiv(N, ch) == k && (best < 0 || c < best)) best = c;
    }
    return best;
  };
  const bool square = least(24, 24) * 120 < least(16, 32) * 100;
  *rows = square ? 32 : 24;
  *cols = square ? 32 : 40;
}

template <int MODE, class SH, int WAVES>
static void tb_launch_shape(const TbGeom &g, const TbStep &k, const TbStepF &kf, const void *xin, const float *lin,
                            void *xout, float *lout, hipStream_t st) {
  const dim3 grid((unsigned)g.total), block(SH::NT);
  const bool lam = k.lam != 0.0;
  if constexpr (MODE == TB_F32S) {
    if (g.pace > 0) {
      if (lam) hipLaunchKernelGGL((k_rk4_tb<MODE, true, SH, WAVES, true>), grid, block, 0, st, g, k, kf, xin, lin, xout, lout);
      else hipLaunchKernelGGL((k_rk4_tb<MODE, false, SH, WAVES, true>), grid, block, 0, st, g, k, kf, xin, lin, xout, lout);
      return;
    }
  }
  if (lam) hipLaunchKernelGGL((k_rk4_tb<MODE, true, SH, WAVES, false>), grid, block, 0, st, g, k, kf, xin, lin, xout, lout);
  else hipLaunchKernelGGL((k_rk4_tb<MODE, false, SH, WAVES, false>), grid, block, 0, st, g, k, kf, xin, lin, xout, lout);
}

static cf_status tb_launch_f64(const TbGeom &g, const TbStep &k, const double *xin, double *xout, hipStream_t st) {
  const TbStepF kf{};
  if (g.shape == 0) tb_launch_shape<TB_F64, TbS12x20, 4>(g, k, kf, xin, nullptr, xout, nullptr, st);
  else if (g.shape == 1) tb_launch_shape<TB_F64, TbS14x36, 4>(g, k, kf, xin, nullptr, xout, nullptr, st);
  else if (g.shape == 2) tb_launch_shape<TB_F64, TbS28x36, 4>(g, k, kf, xin, nullptr, xout, nullptr, st);
  else tb_launch_shape<TB_F64, TbS30x68, 4>(g, k, kf, xin, nullptr, xout, nullptr, st);
  CF_LAUNCHED();
  return CF_OK;
}

// The single-precision stencil's scalars: TbStep's RHS coefficients and stage-input
// steps rounded to float.
static TbStepF tb_step_f32(const TbStep &k) {
  TbStepF f;
  for (int s = 0; s < 4; ++s) {
    f.c_h[s] = (float)k.c_h[s];
    f.inv[s] = (float)k.inv[s];
  }
  f.c_m = (float)k.c_m;
  f.lam = (float)k.lam;
  f.dh = (float)k.dh;
  f.dt = (float)k.dt;
  return f;
}

static cf_status tb_launch_f32c(const TbGeom &g, const TbStep &k, const float *xin, const float *lin, float *xout,
                                float *lout, hipStream_t st) {
  const TbStepF kf{};
  if (g.shape == 0) tb_launch_shape<TB_F32C, TbC14x36, 4>(g, k, kf, xin, lin, xout, lout, st);
  else if (g.shape == 1) tb_launch_shape<TB_F32C, TbC28x36, 4>(g, k, kf, xin, lin, xout, lout, st);
  else tb_launch_shape<TB_F32C, TbC22x68, 3>(g, k, kf, xin, lin, xout, lout, st);
  CF_LAUNCHED();
  return CF_OK;
}

static cf_status tb_launch_sa(const TbGeom &g, const TbStep &k, const float *xin, const float *lin, float *xout,
                              float *lout, hipStream_t st) {
  const TbStepF kf = tb_step_f32(k);
  if (g.shape == 0) tb_launch_shape<TB_F32S, TbS12x20, 4>(g, k, kf, xin, lin, xout, lout, st);
  else if (g.shape == 1) tb_launch_shape<TB_F32S, TbS14x36, 4>(g, k, kf, xin, lin, xout, lout, st);
  else if (g.shape == 2) tb_launch_shape<TB_F32S, TbS28x36, 4>(g, k, kf, xin, lin, xout, lout, st);
  else if (g.shape == 3) tb_launch_shape<TB_F32S, TbS30x68, 4>(g, k, kf, xin, lin, xout, lout, st);
  else tb_launch_shape<TB_F32S, TbS15x132, 4>(g, k, kf, xin, lin, xout, lout, st);
  CF_LAUNCHED();
  return CF_OK;
}

// [a, a + na) and [b, b + nb) do not overlap.
static bool disjoint(const void *a, size_t na, const void *b, size_t nb) {
  const char *x = static_cast<const char *>(a), *y = static_cast<const char *>(b);
  return x + na <= y || y + nb <= x;
}
static bool disjoint(const void *a, const void *b, size_t bytes) { return disjoint(a, bytes, b, bytes); }

static cf_status tb_check(const cf_kg_params *p) {
  CF_REQUIRE(p, "null cf_kg_params");
  CF_REQUIRE(valid_N(p->N), "unsupported lattice size N=%lld (even, 4..2048)", (long long)p->N);
  CF_REQUIRE(p->L > 0.0, "box size L must be positive");
  return CF_OK;
}

// The variants' kernels. 22 x 68 regions of two columns per thread for those whose site
// factors fit the registers so (168 of them; fixed curvature, N=300: 296 -> 230 us a step,
// N=256: 173 -> 154); the comoving ones would spill a hundred and take two columns over 28 x
// 36 regions, 512 threads of up to 256 registers (one column of 1024 threads: N=64 11.8
// against 10.9 us, coarse grid 10.8 against 9.3, N=128 40.4 against 38.1, N=384 1051 against
// 1039; for the others at N=128 one column is the faster, 23.1 against 24.0).
template <int VAR>
static void tb_launch_var(const TbGeom &g, const TbStep &k, const double *xin, double *xout, const double *psi,
                          const TbPsi &cp, hipStream_t st) {
  const dim3 grid((unsigned)g.total);
  if (g.shape == 0) {
    hipLaunchKernelGGL((k_rk4_tb_var<VAR, TbC14x36, 4>), grid, dim3(TbC14x36::NT), 0, st, g, k, xin, xout, psi, cp);
  } else if constexpr (VAR == TB_COMOVING || VAR == TB_APPROX_COMOVING) {
    hipLaunchKernelGGL((k_rk4_tb_var<VAR, TbS28x36, 2>), grid, dim3(TbS28x36::NT), 0, st, g, k, xin, xout, psi, cp);
  } else if (g.shape == 1) {
    hipLaunchKernelGGL((k_rk4_tb_var<VAR, TbC28x36, 4>), grid, dim3(TbC28x36::NT), 0, st, g, k, xin, xout, psi, cp);
  } else {
    hipLaunchKernelGGL((k_rk4_tb_var<VAR, TbC22x68, 3>), grid, dim3(TbC22x68::NT), 0, st, g, k, xin, xout, psi, cp);
  }
}

cf_status tb_step_variant(int var, const cf_kg_params *p, double f_a, const double *psi, const double *xin,
                          double *xout, double t, double dt, int chunk, hipStream_t st, const TbPsi *cps) {
  CF_TRY(tb_check(p));
  const bool comoving = var == TB_COMOVING || var == TB_APPROX_COMOVING;
  CF_REQUIRE(var == TB_SQRT_POTENTIAL || (var == TB_FIXED_CURVATURE && psi) ||
                 (comoving && cps && cps->f[0] && cps->f[1] && cps->f[2] && cps->G > 0),
             "tb_step_variant: bad variant");
  const size_t n = 2 * (size_t)p->N * p->N * p->N;
  CF_REQUIRE(xin && xout && disjoint(xin, xout, n * sizeof(double)),
             "temporally blocked variant step: null or overlapping state buffers");
  const int family = var == TB_FIXED_CURVATURE  ? TB_FAM_CURV
                     : var == TB_SQRT_POTENTIAL ? TB_FAM_SQRT
                     : var == TB_COMOVING       ? TB_FAM_COM
                                                : TB_FAM_APX;
  const TbGeom g = tb_plan(family, p->N, chunk, 0, p->N, p->N);
  TbStep k = tb_step_host(p, t, dt);
  k.fa2 = f_a * f_a;
  const TbPsi cp = cps ? *cps : TbPsi{};
  if (var == TB_FIXED_CURVATURE) tb_launch_var<TB_FIXED_CURVATURE>(g, k, xin, xout, psi, cp, st);
  else if (var == TB_SQRT_POTENTIAL) tb_launch_var<TB_SQRT_POTENTIAL>(g, k, xin, xout, psi, cp, st);
  else if (var == TB_COMOVING) tb_launch_var<TB_COMOVING>(g, k, xin, xout, psi, cp, st);
  else tb_launch_var<TB_APPROX_COMOVING>(g, k, xin, xout, psi, cp, st);
  CF_LAUNCHED();
  return CF_OK;
}

// Pacing of the single-precision-stencil kernel per device, lattice size and chunk (ticks
// of the 100 MHz real-time counter per plane iteration; absent or 0: unpaced), set by
// cf_rk4_tb_tune_pace or cf_rk4_tb_set_pace.
static std::mutex g_pace_mu;
using TbPaceKey = std::tuple<int, int64_t, int, int>;  // device, N, chunk, region rows
static std::map<TbPaceKey, int> g_pace;

static cf_status tb_pace_key(const TbGeom &g, TbPaceKey *key) {
  int dev = 0;
  CF_HIP(hipGetDevice(&dev));
  *key = std::make_tuple(dev, g.N, g.A, g.rb);
  return CF_OK;
}
static cf_status tb_pace_lookup(TbGeom &g) {
  TbPaceKey key;
  CF_TRY(tb_pace_key(g, &key));
  std::lock_guard<std::mutex> lock(g_pace_mu);
  const auto it = g_pace.find(key);
  g.pace = it == g_pace.end() ? 0 : it->second;
  return CF_OK;
}
static cf_status tb_pace_store(const TbGeom &g, int pace) {
  TbPaceKey key;
  CF_TRY(tb_pace_key(g, &key));
  std::lock_guard<std::mutex> lock(g_pace_mu);
  g_pace[key] = pace;
  return CF_OK;
}

// Runs and single steps of the compensated storage: FP64 arithmetic (sa = false) or
// the single-precision stencil (sa = true).
static cf_status tb_launch_comp(bool sa, const TbGeom &g, const TbStep &k, const float *xin, const float *lin,
                                float *xout, float *lout, hipStream_t st) {
  return sa ? tb_launch_sa(g, k, xin, lin, xout, lout, st) : tb_launch_f32c(g, k, xin, lin, xout, lout, st);
}

static cf_status tb_run_comp(const char *name, bool sa, const cf_kg_params *p, float *hi, float *lo, double t0,
                             int64_t k0, int64_t n_steps, double dt, int chunk, void *work, hipStream_t st) {
  CF_TRY(tb_check(p));
  const size_t n = 2 * (size_t)p->N * p->N * p->N;
  const size_t wb = 2 * n * sizeof(float) + 2 * TB_ALIGN_SLACK;  // cf_rk4_tb_work_bytes
  CF_REQUIRE(hi && lo && work && disjoint(hi, lo, n * sizeof(float)) &&
                 disjoint(hi, n * sizeof(float), work, wb) && disjoint(lo, n * sizeof(float), work, wb),
             "%s: null or overlapping buffer", name);
  CF_REQUIRE(n_steps >= 0, "%s: negative step count", name);
  TbGeom g = tb_comp_geom(sa, p->N, chunk);
  if (sa) CF_TRY(tb_pace_lookup(g));
  float *his[2] = {hi, same_residue(work, hi)};
  float *los[2] = {lo, same_residue(his[1] + n, lo)};
  for (int64_t s = 0; s < n_steps; ++s) {
    const double t = t0 + static_cast<double>(k0 + s) * dt;
    CF_TRY(tb_launch_comp(sa, g, tb_step_host(p, t, dt), his[s & 1], los[s & 1], his[(s + 1) & 1],
                          los[(s + 1) & 1], st));
  }
  if (n_steps & 1) {
    CF_HIP(hipMemcpyAsync(hi, his[1], n * sizeof(float), hipMemcpyDeviceToDevice, st));
    CF_HIP(hipMemcpyAsync(lo, los[1], n * sizeof(float), hipMemcpyDeviceToDevice, st));
  }
  return CF_OK;
}

static cf_status tb_step_comp(const char *name, bool sa, const cf_kg_params *p, const float *hi_in,
                              const float *lo_in, float *hi_out, float *lo_out, double t, double dt, int chunk,
                              hipStream_t st) {
  CF_TRY(tb_check(p));
  const size_t b = 2 * (size_t)p->N * p->N * p->N * sizeof(float);
  CF_REQUIRE(hi_in && lo_in && hi_out && lo_out, "%s: null buffer", name);
  CF_REQUIRE(disjoint(hi_in, lo_in, b) && disjoint(hi_out, lo_out, b) && disjoint(hi_in, hi_out, b) &&
                 disjoint(hi_in, lo_out, b) && disjoint(lo_in, hi_out, b) && disjoint(lo_in, lo_out, b),
             "%s: overlapping buffers", name);
  TbGeom g = tb_comp_geom(sa, p->N, chunk);
  if (sa) CF_TRY(tb_pace_lookup(g));
  return tb_launch_comp(sa, g, tb_step_host(p, t, dt), hi_in, lo_in, hi_out, lo_out, st);
}

// Ping-pong buffer of the entry point that allocates nothing
// (cf_rk4_run_tb_f64_noalloc): 2 N^3 doubles for N <= CF_NOALLOC_MAX_N, one copy per
// GPU, held until the process ends. In host code `scratch` names a host-side
// stand-in: kernels and copies take the device address from hipGetSymbolAddress.
static __device__ __align__(256) double scratch[2 * CF_NOALLOC_MAX_N * CF_NOALLOC_MAX_N * CF_NOALLOC_MAX_N];

// scratch's device address on each device, looked up once per device with that
// device current.
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[64] = {};

static cf_status scratch_on_current_device(double **out) {
  int dev = 0;
  CF_HIP(hipGetDevice(&dev));
  CF_REQUIRE(dev >= 0 && dev < 64, "cf_rk4_run_tb_f64_noalloc: device ordinal %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *ptr = nullptr;
    CF_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    CF_REQUIRE(ptr, "cf_rk4_run_tb_f64_noalloc: no device address for the scratch buffer");
    g_scratch_ptr[dev] = ptr;
  }
  *out = static_cast<double *>(g_scratch_ptr[dev]);
  return CF_OK;
}

static cf_status tb_step_comp_slab(const char *name, bool sa, const cf_kg_params *p, int64_t n_planes,
                                   const float *hi_in, const float *lo_in, float *hi_out, float *lo_out, double t,
                                   double dt, int chunk, hipStream_t st) {
  CF_TRY(tb_check(p));
  CF_REQUIRE(n_planes >= 1 && n_planes <= p->N, "%s: n_planes=%lld outside 1..N", name, (long long)n_planes);
  const int64_t NA = n_planes + 2 * TB_GHOST;
  const size_t b = 2 * (size_t)NA * p->N * p->N * sizeof(float);
  CF_REQUIRE(hi_in && lo_in && hi_out && lo_out, "%s: null buffer", name);
  CF_REQUIRE(disjoint(hi_in, lo_in, b) && disjoint(hi_out, lo_out, b) && disjoint(hi_in, hi_out, b) &&
                 disjoint(hi_in, lo_out, b) && disjoint(lo_in, hi_out, b) && disjoint(lo_in, lo_out, b),
             "%s: overlapping buffers", name);
  TbGeom g = tb_plan(sa ? TB_FAM_F32S : TB_FAM_F32C, p->N, chunk, TB_GHOST, TB_GHOST + n_planes, NA);
  if (sa) {
    // The pace tuned for this lattice size and chunk, if any. Its ticks are those of a plane
    // of the whole lattice's regions, so a paced slab runs over the same.
    TbGeom whole = tb_plan_search(TB_FAM_F32S, p->N, g.A, 0, p->N, p->N);  // (leaves the slab's plan kept)
    CF_TRY(tb_pace_lookup(whole));
    if (whole.pace > 0) {
      g = tb_geom(TB_FAM_F32S, whole.shape, p->N, g.A, TB_GHOST, TB_GHOST + n_planes, NA);
      g.pace = whole.pace;
    }
  }
  return tb_launch_comp(sa, g, tb_step_host(p, t, dt), hi_in, lo_in, hi_out, lo_out, st);
}

}  // namespace cf

using namespace cf;

extern "C" {

size_t cf_rk4_tb_work_bytes(int64_t N, int precision) {
  if (!valid_N(N)) return 0;
  const size_t n = 2 * (size_t)N * N * N;
  return (precision == CF_PREC_F32C || precision == CF_PREC_F32S) ? 2 * n * sizeof(float) + 2 * TB_ALIGN_SLACK : n * sizeof(double);
}

cf_status cf_rk4_run_tb_f64(const cf_kg_params *p, double *x, double t0, int64_t k0, int64_t n_steps, double dt,
                            int chunk, void *work, cf_stream stream) {
  CF_TRY(tb_check(p));
  CF_REQUIRE(x && work && disjoint(x, work, 2 * (size_t)p->N * p->N * p->N * sizeof(double)),
             "cf_rk4_run_tb_f64: null or overlapping buffer");
  CF_REQUIRE(n_steps >= 0, "cf_rk4_run_tb_f64: negative step count");
  const TbGeom g = tb_f64_geom(p->N, chunk);
  double *bufs[2] = {x, (double *)work};
  for (int64_t s = 0; s < n_steps; ++s) {
    const double t = t0 + static_cast<double>(k0 + s) * dt;
    CF_TRY(tb_launch_f64(g, tb_step_host(p, t, dt), bufs[s & 1], bufs[(s + 1) & 1], S(stream)));
  }
  if (n_steps & 1) {
    const size_t bytes = 2 * (size_t)p->N * p->N * p->N * sizeof(double);
    CF_HIP(hipMemcpyAsync(x, work, bytes, hipMemcpyDeviceToDevice, S(stream)));
  }
  return CF_OK;
}

cf_status cf_rk4_run_tb_f64_noalloc(const cf_kg_params *p, double *x, double t0, int64_t k0, int64_t n_steps,
                                    double dt, int chunk, cf_stream stream) {
  CF_TRY(tb_check(p));
  CF_REQUIRE(p->N <= CF_NOALLOC_MAX_N,
             "cf_rk4_run_tb_f64_noalloc: N=%lld exceeds the preallocated buffer (N <= %d); use cf_rk4_run_tb_f64",
             (long long)p->N, CF_NOALLOC_MAX_N);
  CF_REQUIRE(x, "cf_rk4_run_tb_f64_noalloc: null state");
  CF_REQUIRE(n_steps >= 0, "cf_rk4_run_tb_f64_noalloc: negative step count");
  double *work = nullptr;
  CF_TRY(scratch_on_current_device(&work));
  const size_t bytes = 2 * (size_t)p->N * p->N * p->N * sizeof(double);
  CF_REQUIRE(disjoint(x, work, bytes), "cf_rk4_run_tb_f64_noalloc: the state overlaps the library's buffer");
  const TbGeom g = tb_f64_geom(p->N, chunk);
  double *bufs[2] = {x, work};
  for (int64_t s = 0; s < n_steps; ++s) {
    const double t = t0 + static_cast<double>(k0 + s) * dt;
    CF_TRY(tb_launch_f64(g, tb_step_host(p, t, dt), bufs[s & 1], bufs[(s + 1) & 1], S(stream)));
  }
  if (n_steps & 1) CF_HIP(hipMemcpyAsync(x, work, bytes, hipMemcpyDeviceToDevice, S(stream)));
  return CF_OK;
}

cf_status cf_rk4_run_tb_f32c(const cf_kg_params *p, float *hi, float *lo, double t0, int64_t k0, int64_t n_steps,
                             double dt, int chunk, void *work, cf_stream stream) {
  return tb_run_comp("cf_rk4_run_tb_f32c", false, p, hi, lo, t0, k0, n_steps, dt, chunk, work, S(stream));
}

cf_status cf_rk4_run_tb_f32s(const cf_kg_params *p, float *hi, float *lo, double t0, int64_t k0, int64_t n_steps,
                             double dt, int chunk, void *work, cf_stream stream) {
  return tb_run_comp("cf_rk4_run_tb_f32s", true, p, hi, lo, t0, k0, n_steps, dt, chunk, work, S(stream));
}

cf_status cf_rk4_step_tb_f64(const cf_kg_params *p, const double *x_in, double *x_out, double t, double dt,
                             int chunk, cf_stream stream) {
  CF_TRY(tb_check(p));
  const size_t n = 2 * (size_t)p->N * p->N * p->N;
  CF_REQUIRE(x_in && x_out && disjoint(x_in, x_out, n * sizeof(double)),
             "cf_rk4_step_tb_f64: null or overlapping state buffers");
  const TbGeom g = tb_f64_geom(p->N, chunk);
  return tb_launch_f64(g, tb_step_host(p, t, dt), x_in, x_out, S(stream));
}

cf_status cf_rk4_step_tb_f64_slab(const cf_kg_params *p, int64_t n_planes, const double *x_in, double *x_out,
                                  double t, double dt, int chunk, cf_stream stream) {
  CF_TRY(tb_check(p));
  CF_REQUIRE(n_planes >= 1 && n_planes <= p->N, "cf_rk4_step_tb_f64_slab: n_planes=%lld outside 1..N",
             (long long)n_planes);
  const int64_t NA = n_planes + 2 * TB_GHOST;  // own planes and four ghost planes on each side
  const size_t bytes = 2 * (size_t)NA * p->N * p->N * sizeof(double);
  CF_REQUIRE(x_in && x_out && disjoint(x_in, x_out, bytes), "cf_rk4_step_tb_f64_slab: null or overlapping slabs");
  // A unit's stored sites depend on planes a0 - 2 .. a1 + 1 of its chunk, all inside the
  // slab for chunks within [4, 4 + n_planes); it loads no plane but those and the two after
  // them, and its lattice offsets wrap at NA.
  const TbGeom g = tb_plan(TB_FAM_F64, p->N, chunk, TB_GHOST, TB_GHOST + n_planes, NA);
  return tb_launch_f64(g, tb_step_host(p, t, dt), x_in, x_out, S(stream));
}

cf_status cf_rk4_step_tb_f32c(const cf_kg_params *p, const float *hi_in, const float *lo_in, float *hi_out,
                              float *lo_out, double t, double dt, int chunk, cf_stream stream) {
  return tb_step_comp("cf_rk4_step_tb_f32c", false, p, hi_in, lo_in, hi_out, lo_out, t, dt, chunk, S(stream));
}

cf_status cf_rk4_step_tb_f32s(const cf_kg_params *p, const float *hi_in, const float *lo_in, float *hi_out,
                              float *lo_out, double t, double dt, int chunk, cf_stream stream) {
  return tb_step_comp("cf_rk4_step_tb_f32s", true, p, hi_in, lo_in, hi_out, lo_out, t, dt, chunk, S(stream));
}

cf_status cf_rk4_step_tb_f32c_slab(const cf_kg_params *p, int64_t n_planes, const float *hi_in, const float *lo_in,
                                   float *hi_out, float *lo_out, double t, double dt, int chunk, cf_stream stream) {
  return tb_step_comp_slab("cf_rk4_step_tb_f32c_slab", false, p, n_planes, hi_in, lo_in, hi_out, lo_out, t, dt, chunk,
                           S(stream));
}

cf_status cf_rk4_step_tb_f32s_slab(const cf_kg_params *p, int64_t n_planes, const float *hi_in, const float *lo_in,
                                   float *hi_out, float *lo_out, double t, double dt, int chunk, cf_stream stream) {
  return tb_step_comp_slab("cf_rk4_step_tb_f32s_slab", true, p, n_planes, hi_in, lo_in, hi_out, lo_out, t, dt, chunk,
                           S(stream));
}

// Pacing of the single-precision-stencil step: time the step of this lattice at a
// range of paces and keep one with margin. Where pacing helps, the rate falls below the
// fastest pace and declines slowly above it, and where the fall begins moves with the
// clock, so each pace P is scored by the slowest of P - TB_PACE_MARGIN .. P, and the best
// score wins (at equal scores the larger pace); unpaced wins if it is as fast. With the
// 24 x 40 regions and the halo of four that the kernel had before, pacing gave 101 -> 109
// GSite*step/s at N=512; the large regions drift less and gain little or nothing.
constexpr int TB_PACE_MARGIN = 2;

// Chunk lengths within this many percent of the cost model's best that the pace tuner
// tries when the caller leaves the chunk to it, the cheapest TB_CHUNK_NEAR_MAX of them.
constexpr int TB_CHUNK_NEAR_PCT = 5;
constexpr size_t TB_CHUNK_NEAR_MAX = 4;

// Pace of launches over geometry g: the pick and its score (the slowest ms per step over
// the picked pace and the TB_PACE_MARGIN paces below it; the unpaced ms for pick 0).
static cf_status tb_tune_pace_geom(TbGeom g, const TbStep &k, const float *hi, const float *lo, float *ho,
                                   float *lw, hipStream_t st, hipEvent_t e0, hipEvent_t e1, int *pick_out,
                                   float *score_out) {
  std::map<int, float> ms;  // pace -> ms per step
  auto time_pace = [&](int pace) -> cf_status {
    if (ms.count(pace)) return CF_OK;
    g.pace = pace;
    CF_TRY(tb_launch_sa(g, k, hi, lo, ho, lw, st));  // warm-up
    float best = 1e30f;
    for (int w = 0; w < 2; ++w) {  // the faster of two windows of three launches
      CF_HIP(hipEventRecord(e0, st));
      for (int r = 0; r < 3; ++r) CF_TRY(tb_launch_sa(g, k, hi, lo, ho, lw, st));
      CF_HIP(hipEventRecord(e1, st));
      CF_HIP(hipEventSynchronize(e1));
      float el = 0.0f;
      CF_HIP(hipEventElapsedTime(&el, e0, e1));
      best = el / 3.0f < best ? el / 3.0f : best;
    }
    ms[pace] = best;
    return CF_OK;
  };
  // coarse grid 0.64 .. 3.2 us per plane, then every tick from below the coarse best to
  // the margin above it
  for (int pace = 0; pace <= 320; pace += (pace == 0 ? 64 : 8)) CF_TRY(time_pace(pace));
  int coarse = 0;
  for (const auto &kv : ms)
    if (kv.second < ms[coarse]) coarse = kv.first;
  if (coarse > 0)
    for (int pace = coarse - 8; pace <= coarse + 8 + TB_PACE_MARGIN; ++pace) CF_TRY(time_pace(pace));
  int pick = 0;
  float pick_worst = ms[0];
  for (const auto &kv : ms) {
    if (kv.first - TB_PACE_MARGIN < 1) continue;
    float worst = 0.0f;
    bool full = true;
    for (int q = kv.first - TB_PACE_MARGIN; q <= kv.first && full; ++q) {
      const auto it = ms.find(q);
      full = it != ms.end();
      if (full) worst = it->second > worst ? it->second : worst;
    }
    if (full && worst <= pick_worst && (pick > 0 || worst < ms[0])) {
      pick = kv.first;
      pick_worst = worst;
    }
  }
  *pick_out = pick;
  *score_out = pick_worst;
  return CF_OK;
}

cf_status cf_rk4_tb_tune_pace(const cf_kg_params *p, const float *hi, const float *lo, double t, double dt, int chunk,
                              void *work, cf_stream stream, int *pace_out) {
  CF_TRY(tb_check(p));
  const size_t n = 2 * (size_t)p->N * p->N * p->N;
  const size_t wb = 2 * n * sizeof(float) + 2 * TB_ALIGN_SLACK;  // cf_rk4_tb_work_bytes
  CF_REQUIRE(hi && lo && work && disjoint(hi, lo, n * sizeof(float)) &&
                 disjoint(hi, n * sizeof(float), work, wb) && disjoint(lo, n * sizeof(float), work, wb),
             "cf_rk4_tb_tune_pace: null or overlapping buffer");
  hipStream_t st = S(stream);
  std::vector<int> chunks;
  if (chunk > 0)
    chunks.push_back(chunk);
  else
    (void)tb_plan_search(TB_FAM_F32S, p->N, 0, 0, p->N, p->N, &chunks, TB_CHUNK_NEAR_PCT);
  if (chunks.size() > TB_CHUNK_NEAR_MAX) chunks.resize(TB_CHUNK_NEAR_MAX);
  float *ho = same_residue(work, hi), *lw = same_residue(ho + n, lo);
  const TbStep k = tb_step_host(p, t, dt);
  hipEvent_t e0 = nullptr, e1 = nullptr;
  CF_HIP(hipEventCreate(&e0));
  if (hipEventCreate(&e1) != hipSuccess) {
    (void)hipEventDestroy(e0);
    CF_REQUIRE(false, "cf_rk4_tb_tune_pace: hipEventCreate failed");
  }
  cf_status rc = CF_OK;
  std::vector<TbGeom> picks;
  for (size_t i = 0; i < chunks.size() && rc == CF_OK; ++i) {
    TbGeom g = tb_plan(TB_FAM_F32S, p->N, chunks[i], 0, p->N, p->N);
    float score = 0.0f;
    rc = tb_tune_pace_geom(g, k, hi, lo, ho, lw, st, e0, e1, &g.pace, &score);
    if (rc == CF_OK) rc = tb_pace_store(g, g.pace);
    picks.push_back(g);
  }
  // Between chunks: each at its pick, timed again over longer windows (the fastest of
  // three windows of five launches; a pace tuning's short windows and margin rank the
  // paces of one chunk, not chunks whose rate curves differ in steepness).
  auto time_pick = [&](const TbGeom &g, float *ms) -> cf_status {
    *ms = 1e30f;
    for (int w = 0; w < 3; ++w) {
      CF_TRY(tb_launch_sa(g, k, hi, lo, ho, lw, st));  // a gap-free start for the window
      CF_HIP(hipEventRecord(e0, st));
      for (int r = 0; r < 5; ++r) CF_TRY(tb_launch_sa(g, k, hi, lo, ho, lw, st));
      CF_HIP(hipEventRecord(e1, st));
      CF_HIP(hipEventSynchronize(e1));
      float el = 0.0f;
      CF_HIP(hipEventElapsedTime(&el, e0, e1));
      if (el / 5.0f < *ms) *ms = el / 5.0f;
    }
    return CF_OK;
  };
  int best_chunk = 0, best_pace = 0;
  float best_ms = 0.0f;
  for (size_t i = 0; i < picks.size() && rc == CF_OK && chunks.size() > 1; ++i) {
    float ms = 0.0f;
    rc = time_pick(picks[i], &ms);
    if (rc == CF_OK && (i == 0 || ms < best_ms)) {
      best_chunk = picks[i].A;
      best_pace = picks[i].pace;
      best_ms = ms;
    }
  }
  if (chunks.size() == 1 && rc == CF_OK) {
    best_chunk = picks[0].A;
    best_pace = picks[0].pace;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  CF_TRY(rc);
  if (chunk <= 0) {
    int dev = 0;
    CF_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_chunk_mu);
    g_chunk[std::make_pair(dev, p->N)] = best_chunk;
  }
  if (pace_out) *pace_out = best_pace;
  return CF_OK;
}

cf_status cf_rk4_tb_set_pace(int64_t N, int chunk, int pace) {
  CF_REQUIRE(valid_N(N), "cf_rk4_tb_set_pace: unsupported lattice size N=%lld", (long long)N);
  CF_REQUIRE(pace >= 0 && pace <= 100000, "cf_rk4_tb_set_pace: pace %d outside 0..100000", pace);
  return tb_pace_store(tb_comp_geom(true, N, chunk), pace);
}

cf_status cf_rk4_tb_set_chunk(int64_t N, int chunk) {
  CF_REQUIRE(valid_N(N), "cf_rk4_tb_set_chunk: unsupported lattice size N=%lld", (long long)N);
  CF_REQUIRE(chunk >= 0 && chunk <= N, "cf_rk4_tb_set_chunk: chunk %d outside 0..N", chunk);
  int dev = 0;
  CF_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_chunk_mu);
  if (chunk == 0)
    g_chunk.erase(std::make_pair(dev, N));
  else
    g_chunk[std::make_pair(dev, N)] = chunk;
  return CF_OK;
}

int cf_rk4_tb_get_chunk(int64_t N) {
  if (!valid_N(N)) return -1;
  return tb_comp_geom(true, N, 0).A;
}

cf_status cf_rk4_tb_f32s_region(int64_t N, int *rows, int *cols) {
  CF_REQUIRE(valid_N(N), "cf_rk4_tb_f32s_region: unsupported lattice size N=%lld", (long long)N);
  CF_REQUIRE(rows && cols, "cf_rk4_tb_f32s_region: null output");
  tb_f32s_class(N, rows, cols);
  return CF_OK;
}

cf_status cf_rk4_tb_geometry(int64_t N, int precision, int chunk, int geom[6]) {
  CF_REQUIRE(valid_N(N), "cf_rk4_tb_geometry: unsupported lattice size N=%lld", (long long)N);
  CF_REQUIRE(precision == CF_PREC_F64 || precision == CF_PREC_F32C || precision == CF_PREC_F32S,
             "cf_rk4_tb_geometry: unknown precision %d", precision);
  CF_REQUIRE(geom, "cf_rk4_tb_geometry: null output");
  const TbGeom g = precision == CF_PREC_F64 ? tb_f64_geom(N, chunk) : tb_comp_geom(precision == CF_PREC_F32S, N, chunk);
  const int v[6] = {g.rb, g.rc, g.Tb, g.Tc, g.A, g.total};
  for (int i = 0; i < 6; ++i) geom[i] = v[i];
  return CF_OK;
}

int cf_rk4_tb_get_pace(int64_t N, int chunk) {
  if (!valid_N(N)) return -1;
  TbGeom g = tb_comp_geom(true, N, chunk);
  if (tb_pace_lookup(g) != CF_OK) return -1;
  return g.pace;
}

}  // extern "C"
