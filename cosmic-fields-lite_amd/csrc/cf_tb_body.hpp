// cf_tb_body.hpp -- the temporally blocked RK4 step of one work unit (an output
// tile of one lattice over a chunk of a-planes), shared by the single-lattice and
// variant kernels (cf_rk4_tb.hip) and the ensemble kernels (cf_ensemble.hip).
//
// Domain of dependence. With dphi/dt = pi, phi of every stage input is local in the
// stage before it: y1.phi = x.phi + h/2 x.pi, y2.phi = x.phi + h/2 y1.pi and
// y3.phi = x.phi + h y2.pi; only dpi/dt has a stencil, and of phi alone. So k1 and k2
// at a site need x within distance 1 (their stencils run over x.phi and y1.phi), they
// give y2.phi and y3.phi there, and k3 and k4 need those within distance 1: the whole
// step reaches two sites, not one per stage, and two stencils run side by side.
//
// Geometry. A block covers an RB x RC (b, c) region of the lattice: an output tile of
// T x Tc sites plus a halo of two sites on every side. Each thread owns VC (1 or 2)
// neighbouring columns of a row and marches along a through the chunk's planes
// [a0, a1), keeping in registers the planes the stencils need along a:
//
//   iteration j takes x at plane P = a0 - 2 + j (loaded two iterations ahead) and y1.phi
//     A at P-1 (needs x.phi, y1.phi at P-2..P)     -> k1, k2; y2.phi, y3.phi, partial sums
//     B at P-2 (needs y2.phi, y3.phi at P-3..P-1)  -> k3, k4; new state at P-2
//
// The first stored plane is that of j = 4 and needs A from j = 2 on: the loop starts there,
// with the first two planes taken straight from their loads, and iterations 2 and 3 leave
// B out. So a chunk of A planes takes A + 2 iterations, two of them half. (Running all
// stages from j = 0: A + 4 full iterations; N=32 5.6 against 3.6 us, N=64 7.8 / 6.0,
// N=128 19.4 / 17.7.) The in-plane neighbours come from four
// plane buffers in LDS (x.phi, y1.phi of P-1; y2.phi, y3.phi of P-2), all known when the
// iteration starts: they are written together, and with two sets of buffers one barrier
// per plane suffices. The histories are three planes deep; the loop is unrolled by six
// (three phases times two buffer sets), so advancing a plane renames registers. Per plane
// and site the FP64 step then issues its 80 additions and multiplications and nothing
// else on the vector unit (one stage per plane with a halo of four sites issued 108 for
// 1.78 region sites per output site against 1.23-1.31 here).
//
// Memory. Loads and stores go through buffer resources over one plane, VC values each
// (16 bytes in FP64), with per-lane offsets that never change: lanes outside the tile
// hold an offset past the plane's end, so no branch surrounds a memory operation (before
// j = 4 the lo parts are read through an empty resource). N is even, so a pair of columns
// never straddles the periodic wrap. The plane loads are issued two iterations
// ahead; the barrier is a bare s_barrier after a wait for this wavefront's LDS operations,
// so it waits for no load. What bounds it: at N=512 the bytes moved, 4.8 TB/s of the 32
// it cannot do without (a plain copy reaches 4.8-5.0 on this part); below N=200 vector
// and LDS issue and the chain of dependent FP64 operations of a plane.
//
// Tiles. Tc is 16, 32, 64 or 128 in the single-lattice shapes (N where that is smaller), so
// that a tile's rows begin and end on 128-byte lines where the lattice's rows do: 28 x 28
// tiles (32 x 32 regions), whose row ends share lines with their neighbours, ran at 98
// GSite*step/s at N=512 in FP64 against 134 for 24 x 32 tiles and 150 for 26 x 64. (Ensembles
// that fit the cache may take 28 x 28 or 20 x 36 ones.) T may be less than the region's rows
// hold, for more and smaller tiles.
//
// Arithmetic. Per site and stage the operations, their order and their rounding are
// those of the fused stage kernels (cf_stencil.hip): FP64 keeps acc = 1*x + dt/6 k1
// + dt/3 k2 + dt/3 k3 and ends with acc + dt/6 k4; TB_F32C (compensated FP32 storage)
// rounds y and the increment D to float after every stage and folds (hi + lo) +
// (D + dt/6 k4) in double. The results are therefore bit-identical to the four-kernel
// path. TB_F32S (compensated storage, single-precision stencil): each stage's force is
// float arithmetic on the float stage inputs, y = fma(c, k, hi) in float, the increment
// D is kept unrounded in double (D = fma(dt/3, k, D)) and the new state is (hi + lo) +
// fma(dt/6, k4, D). That scheme has no four-kernel form; the oracle restates it
// (orc_rk4_step_f32s).
#pragma once

#include <type_traits>

#include "cf_common.hpp"

namespace cf {

constexpr int TBH = 2;        // halo of a region: the step's domain of dependence
constexpr int TB_GHOST = 4;   // ghost planes of a slab buffer on each side (two are read)

enum : int { TB_F64 = 0, TB_F32C = 1, TB_F32S = 2 };  // arithmetic and storage (= CF_PREC_*)

// A region shape: rows x columns, columns per thread, threads per block. Threads past
// the region's rows extend it by further rows that store nothing.
template <int RB_, int RC_, int VC_, int NT_>
struct TbShape {
  static constexpr int RB = RB_, RC = RC_, VC = VC_, NT = NT_;
  static constexpr int TPR = RC / VC;                // threads per row
  static constexpr int ROWS = (NT + TPR - 1) / TPR;  // rows of a plane buffer
  static constexpr int PLANE = ROWS * RC;
  static constexpr int LDS = 8 * PLANE + 2 * RC;     // elements: two sets of four planes, a row before and after
  static_assert(RC % VC == 0 && RB > 2 * TBH && RC > 2 * TBH && RB * TPR <= NT && NT % 64 == 0, "region shape");
};

// Scalars of one step: per stage (-3H) and inv_ah_sqr at the stage time, and
// the step's constants.
struct TbStep {
  double c_h[4], inv[4];
  double c_m, lam, dh, dt, dt6, dt3;
  double m, fa2;  // equation variants: mass, f_a^2
};

// The scalars of the single-precision stencil (the compensated mode with float
// right-hand sides): the RHS coefficients and the stage-input step lengths of
// TbStep, rounded to float. The increment weights dt/6, dt/3 stay double.
struct TbStepF {
  float c_h[4], inv[4];
  float c_m, lam, dh, dt;
};

// Equation of the step body: the Klein-Gordon family (+ lambda phi^3), or the
// fixed-curvature / sqrt-potential variants in the operation order of their CUDA
// kernels (Fixed_Curvature_FRW_equation_kernel, equations_cuda.cu:114-137;
// Sqrt_Potential_FRW_equation_kernel, :83-106), as in csrc/cf_variants.hip.
enum : int { TB_KG = 0, TB_FIXED_CURVATURE = 1, TB_SQRT_POTENTIAL = 2, TB_COMOVING = 3, TB_APPROX_COMOVING = 4 };

// Comoving curvature: Psi | dPsi/dt ([Psi (G^3) | dPsi (G^3)]) at the step's three
// stage times (0: t, 1: t + dt/2 for stages 2 and 3, 2: t + dt); G = N (TB_COMOVING)
// or the coarse grid M (TB_APPROX_COMOVING, site (a,b,c) reads cell
// ((x + hs) % N) / sd per axis, sd = N / M, hs = sd / 2).
struct TbPsi {
  const double *f[3];
  int64_t G, sd, hs;
};

// Pacing. Neighbouring tiles read each other's edge rows and columns of every plane;
// those reads hit the L2 only while the two blocks march through the same planes at
// about the same time. Blocks that start together drift apart once an iteration's
// compute is short against its memory latency, and their halo reads then go to HBM.
// With PACE every wavefront of a block waits, before the barrier of iteration j, until
// pace * j ticks of the 100 MHz real-time counter have passed since the block began,
// so blocks cannot run ahead of the schedule (blocks that fall behind it catch up at
// full speed). Pacing changes timing only, never results.

// One work unit: lattice size, output tile origin and edges (T along b, Tc along
// c), plane chunk, and the planes NA that the state buffers hold along a (N for a
// periodic lattice; a slab of a larger lattice holds its planes plus ghost planes,
// and the unit's planes stay within it). Plane indices wrap at NA.
struct TbUnit {
  int64_t N;
  int64_t b0, c0, a0, a1;
  int T, Tc;
  int64_t NA;
  int pace;  // ticks per plane iteration (bodies built with PACE; see Pacing above)
};

__device__ __forceinline__ double tb_rhs(double phi, double pa1, double pam, double pb1, double pbm, double pc1,
                                         double pcm, double pi, double c_h, double c_m, double lam, double inv,
                                         bool has_lam) {
  double v = c_h * pi - c_m * phi;
  if (has_lam) v = v - ((lam * phi) * phi) * phi;
  double r = v + inv * ((((-6.0 * phi + pa1) + pam) + pb1) + pbm);
  return r + inv * (pc1 + pcm);
}

// The Klein-Gordon force in float (single-precision stencil): the seven-point sum
// in one chain (a, b, c neighbours; -6 phi + phi_a+ fused), then inv_ah_sqr times the
// sum fused onto (-3H) pi - m^2 phi (itself one fused multiply-add).
template <bool LAM>
__device__ __forceinline__ float tb_rhs_f32(float phi, float pa1, float pam, float pb1, float pbm, float pc1,
                                            float pcm, float pi, float c_h, float c_m, float lam, float inv) {
  float v = __builtin_fmaf(c_h, pi, -(c_m * phi));
  if constexpr (LAM) v = __builtin_fmaf(-((lam * phi) * phi), phi, v);
  const float s7 = ((((__builtin_fmaf(-6.0f, phi, pa1) + pam) + pb1) + pbm) + pc1) + pcm;
  return __builtin_fmaf(inv, s7, v);
}

// What the variants' forces read at a site besides phi and pi: (e^{2Psi} m) m, e^{4Psi}
// (their Taylor forms on the coarse grid) and 4 dPsi/dt. They depend on the stage time
// alone, so stages that share a time share them: two exponentials per site and time
// instead of two per site and stage.
struct TbSite {
  double em, e4, dp4;
};
template <int VAR>
__device__ __forceinline__ TbSite tb_site(double ps, double dp, double m) {
  TbSite s{0.0, 0.0, 0.0};
  if constexpr (VAR == TB_FIXED_CURVATURE || VAR == TB_COMOVING) {
    s.em = (exp(2.0 * ps) * m) * m;
    s.e4 = exp(4.0 * ps);
    s.dp4 = 4.0 * dp;
  } else if constexpr (VAR == TB_APPROX_COMOVING) {
    s.em = (((1.0 + 2.0 * ps) + (2.0 * ps) * ps) * m) * m;
    s.e4 = (1.0 + 4.0 * ps) + (8.0 * ps) * ps;
    s.dp4 = 4.0 * dp;
  }
  return s;
}

template <int VAR, bool LAM>
__device__ __forceinline__ double tb_force(double phi, double pa1, double pam, double pb1, double pbm, double pc1,
                                           double pcm, double pi, double c_h, double inv, const TbStep &k,
                                           const TbSite &s) {
  if constexpr (VAR == TB_KG) {
    return tb_rhs(phi, pa1, pam, pb1, pbm, pc1, pcm, pi, c_h, k.c_m, k.lam, inv, LAM);
  } else if constexpr (VAR == TB_FIXED_CURVATURE) {
    const double s7 = (((((-6.0 * phi + pa1) + pam) + pb1) + pbm) + pc1) + pcm;
    return (c_h * pi - s.em * phi) + (s.e4 * inv) * s7;
  } else if constexpr (VAR == TB_COMOVING) {
    const double ci = s.e4 * inv;
    const double v = ((c_h + s.dp4) * pi - s.em * phi) + ci * ((((-6.0 * phi + pa1) + pam) + pb1) + pbm);
    return v + ci * (pc1 + pcm);
  } else if constexpr (VAR == TB_APPROX_COMOVING) {
    const double s7 = (((((-6.0 * phi + pa1) + pam) + pb1) + pbm) + pc1) + pcm;
    return ((c_h + s.dp4) * pi - s.em * phi) + (s.e4 * inv) * s7;
  } else {
    const double s7 = (((((-6.0 * phi + pa1) + pam) + pb1) + pbm) + pc1) + pcm;
    return (c_h * pi - (k.c_m * phi) / sqrt(1.0 + (phi * phi) / k.fa2)) + inv * s7;
  }
}

// Buffer-resource access to one lattice plane (gfx9 raw buffer, stride 0,
// num_records = plane bytes; word 3 = 0x00020000 as for all gfx9 parts). An
// offset of TB_OOB is out of range: stores to it are dropped, loads return 0.
constexpr uint32_t TB_OOB = 0x80000000u;
typedef unsigned int tb_u2 __attribute__((ext_vector_type(2)));
typedef unsigned int tb_u4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t tb_plane(const void *base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, bytes, 0x00020000);
}
// VC neighbouring columns of one row.
template <class T, int V>
struct TbVec {
  T v[V];
};
template <class T, int V>
__device__ __forceinline__ TbVec<T, V> tb_load(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  typedef TbVec<T, V> R;
  if constexpr (sizeof(R) == 16) return __builtin_bit_cast(R, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
  else if constexpr (sizeof(R) == 8) return __builtin_bit_cast(R, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
  else return __builtin_bit_cast(R, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
}
template <class T, int V>
__device__ __forceinline__ void tb_store(const TbVec<T, V> &v, __amdgpu_buffer_rsrc_t r, uint32_t off) {
  if constexpr (sizeof(v) == 16) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(tb_u4, v), r, (int)off, 0, 0);
  else if constexpr (sizeof(v) == 8) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(tb_u2, v), r, (int)off, 0, 0);
  else __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, v), r, (int)off, 0, 0);
}

// Workgroup barrier for the plane buffers: this wavefront's LDS operations complete
// (lgkmcnt 0), then s_barrier; vector memory operations stay in flight. The empty asm
// statements keep the compiler from moving memory operations across it.
__device__ __forceinline__ void tb_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int N>
struct tb_ic {
  static constexpr int value = N;
};

// The element type of the plane buffers and histories. In the compensated modes every
// carried value is exactly representable in float; WIDE (TB_F32C, one column per thread)
// holds it widened, so that each is converted once and not at every neighbour's read
// (N=128: 24.1 against 24.9 us a step); two columns per thread have no registers for
// that (26 x 64 tiles of float histories: N=512 1019 against 1052 us).
template <int MODE, class SH>
using TbElem = std::conditional_t<MODE == TB_F64 || (MODE == TB_F32C && SH::VC == 1), double, float>;

// One unit. smem: SH::LDS elements of TbElem, 16-byte aligned; a caller that runs several
// units in a row must barrier between them. xin / xout: the state (TB_F64, doubles) or
// its hi parts (floats), lin / lout: the lo parts.
template <int MODE, bool LAM, class SH, int VAR = TB_KG, bool PACE = false>
__device__ __forceinline__ void tb_unit(void *smem, const TbUnit &u, const TbStep &k, const TbStepF &kf,
                                        const void *xin_, const float *lin, void *xout_, float *lout,
                                        const double *psi = nullptr, const TbPsi cps = TbPsi{}) {
  static_assert(VAR == TB_KG || MODE == TB_F64, "the equation variants are FP64");
  constexpr int VC = SH::VC, RC = SH::RC, PL = SH::PLANE;
  typedef std::conditional_t<MODE == TB_F64, double, float> T;   // storage
  typedef TbElem<MODE, SH> H;                                    // histories, plane buffers
  typedef std::conditional_t<MODE == TB_F32S, float, double> Av; // force arithmetic
  typedef std::conditional_t<MODE == TB_F32S, double, T> Dv;     // partial sum / increment
  typedef TbVec<T, VC> V;
  typedef TbVec<H, VC> HV;
  const T *xin = (const T *)xin_;
  T *xout = (T *)xout_;
  H *lds = (H *)smem;
  const int tid = (int)threadIdx.x;
  const int r = tid / SH::TPR, cc = (tid % SH::TPR) * VC;
  const int N = (int)u.N;
  const int64_t NN = u.N * u.N, N3 = NN * u.NA;  // N3: offset of the pi planes
  const int plane_bytes = (int)(NN * (int64_t)sizeof(T));
  int b = ((int)u.b0 - TBH + r) % N;
  if (b < 0) b += N;
  int c = ((int)u.c0 - TBH + cc) % N;
  if (c < 0) c += N;
  const uint32_t ld_off = (uint32_t)(b * N + c) * (uint32_t)sizeof(T);
  const bool out_ok = r >= TBH && r < TBH + u.T && (int)u.b0 + (r - TBH) < N && cc >= TBH && cc < TBH + u.Tc &&
                      (int)u.c0 + (cc - TBH) < N;
  const uint32_t st_off = out_ok ? ld_off : TB_OOB;
  // own slot of plane buffer 0; the rows above and below are RC away (the region's edge
  // rows and columns read a neighbouring buffer's values or the spare rows: their results
  // reach no stored site)
  H *me = lds + RC + r * RC + cc;

  HV XF[3] = {}, Y1F[3] = {}, Y2F[3] = {}, Y3F[3] = {}, XP[3] = {}, Y2P = {};
  TbVec<Dv, VC> AF = {}, AP = {};
  V LDF[2], LDP[2];
  TbVec<float, VC> LF[2] = {}, LP[2] = {};
  auto wrap = [&](int64_t P) -> int64_t {
    int64_t q = P % u.NA;
    if (q < 0) q += u.NA;
    return q * NN;
  };
  auto next_plane = [&](int64_t off) -> int64_t {
    off += NN;
    return off == N3 ? 0 : off;
  };
  int64_t off_ld = wrap(u.a0 - TBH);  // next plane to load
  int64_t off_st = off_ld;            // plane P-2 of the first iteration, j = 2
  int64_t off_lo = off_st;
  const int iters = (int)(u.a1 - u.a0) + 4;
  auto load = [&](int s) {
    LDF[s] = tb_load<T, VC>(tb_plane(xin + off_ld, plane_bytes), ld_off);
    LDP[s] = tb_load<T, VC>(tb_plane(xin + N3 + off_ld, plane_bytes), ld_off);
    off_ld = next_plane(off_ld);
  };
  // the compensation terms of iteration j's output plane (nothing before j = 4)
  auto load_lo = [&](int s, int j) {
    const int nb = j >= 4 ? plane_bytes : 0;
    LF[s] = tb_load<float, VC>(tb_plane(lin + off_lo, nb), st_off);
    LP[s] = tb_load<float, VC>(tb_plane(lin + N3 + off_lo, nb), st_off);
    off_lo = next_plane(off_lo);
  };
  // x at the planes of j = 0 and 1, then the prefetches of j = 2 and 3
  V first[2][2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    load(q);
    first[q][0] = LDF[q];
    first[q][1] = LDP[q];
  }
  load(0);
  load(1);
  if constexpr (MODE != TB_F64) {
    load_lo(0, 2);
    load_lo(1, 3);
  }
  // Variants: Psi (and dPsi) of A's plane at the stage times of k1 and k2 and of B's plane
  // at that of k4, loaded one iteration ahead; what k3 needs is what k2 had.
  constexpr bool CURV = VAR == TB_FIXED_CURVATURE, COM = VAR == TB_COMOVING, APX = VAR == TB_APPROX_COMOVING;
  const int64_t G3 = APX ? cps.G * cps.G * cps.G : N3;
  const int field_bytes = APX ? (int)(cps.G * cps.G * 8) : plane_bytes;
  uint32_t ps_off[VC] = {};
  int64_t off_a = 0, off_b = 0;        // plane offsets of the next iteration's A and B in Psi's grid
  int rem_a = 0, rem_b = 0;            // APX: planes passed within the coarse plane
  TbVec<double, VC> psA[2] = {}, dpA[2] = {}, psB = {}, dpB = {};
  TbSite site_mid[VC] = {};            // of B's plane, from the iteration before
  if constexpr (CURV || COM) {
    off_a = wrap(u.a0 - 1);
    off_b = wrap(u.a0 - 2);
  } else if constexpr (APX) {
    const int sd = (int)cps.sd, hs = (int)cps.hs;
#pragma unroll
    for (int v = 0; v < VC; ++v)
      ps_off[v] = (uint32_t)((((b + hs) % N) / sd) * (int)cps.G + ((c + v + hs) % N) / sd) * 8u;
    auto cell = [&](int64_t P, int64_t &off, int &rem) {
      const int q = (int)(((P + 2 * u.NA) % u.NA + hs) % u.NA);
      off = (int64_t)(q / sd) * cps.G * cps.G;
      rem = q % sd;
    };
    cell(u.a0 - 1, off_a, rem_a);
    cell(u.a0 - 2, off_b, rem_b);
  }
  auto field = [&](const double *f, int64_t off, uint32_t lane) {
    if constexpr (!APX) return tb_load<double, VC>(tb_plane(f + off, field_bytes), lane);
    TbVec<double, VC> r;
#pragma unroll
    for (int v = 0; v < VC; ++v) r.v[v] = tb_load<double, 1>(tb_plane(f + off, field_bytes), ps_off[v]).v[0];
    return r;
  };
  auto step_cell = [&](int64_t &off, int &rem) {
    if (++rem == (int)cps.sd) {
      rem = 0;
      off += cps.G * cps.G;
      if (off == G3) off = 0;
    }
  };
  auto load_psi = [&]() {
    if constexpr (CURV) {
      psA[0] = field(psi, off_a, ld_off);
      off_a = next_plane(off_a);
    } else if constexpr (COM || APX) {
      psA[0] = field(cps.f[0], off_a, ld_off);
      dpA[0] = field(cps.f[0] + G3, off_a, ld_off);
      psA[1] = field(cps.f[1], off_a, ld_off);
      dpA[1] = field(cps.f[1] + G3, off_a, ld_off);
      psB = field(cps.f[2], off_b, st_off);
      dpB = field(cps.f[2] + G3, off_b, st_off);
      if constexpr (COM) {
        off_a = next_plane(off_a);
        off_b = next_plane(off_b);
      } else {
        step_cell(off_a, rem_a);
        step_cell(off_b, rem_b);
      }
    }
  };
  load_psi();

  // k of one stage at the thread's columns: x0 the stage input's phi at the plane, xa and
  // xm at the planes above and below, pi its pi; bp its own slot in the plane buffer.
  auto force = [&](const HV &x0, const HV &xa, const HV &xm, const HV &pi, const H *bp, int stage,
                   const TbSite (&s)[VC], Av (&out)[VC]) {
    const H nx = bp[VC], pv = bp[-1];
    const HV up = *(const HV *)(bp + RC), dn = *(const HV *)(bp - RC);
#pragma unroll
    for (int v = 0; v < VC; ++v) {
      const H cn = v + 1 < VC ? x0.v[v + 1] : nx, cp = v > 0 ? x0.v[v - 1] : pv;
      if constexpr (MODE == TB_F32S)
        out[v] = tb_rhs_f32<LAM>(x0.v[v], xa.v[v], xm.v[v], up.v[v], dn.v[v], cn, cp, pi.v[v], kf.c_h[stage], kf.c_m,
                                 kf.lam, kf.inv[stage]);
      else
        out[v] = tb_force<VAR, LAM>((double)x0.v[v], (double)xa.v[v], (double)xm.v[v], (double)up.v[v],
                                    (double)dn.v[v], (double)cn, (double)cp, (double)pi.v[v], k.c_h[stage],
                                    k.inv[stage], k, s[v]);
    }
  };
  // a stage input x + c k (rounded to the storage type) and the increment d + c k
  auto input = [&](H x, Av c, Av kk) -> H {
    if constexpr (MODE == TB_F32S) return __builtin_fmaf(c, kk, x);
    else return (H)(T)((double)x + c * kk);
  };
  auto add = [&](Dv d, double c, double kk) -> Dv {
    if constexpr (MODE == TB_F32S) return __builtin_fma(c, kk, d);
    else return (Dv)((double)d + c * kk);
  };
  const Av dh = MODE == TB_F32S ? (Av)kf.dh : (Av)k.dh, dt = MODE == TB_F32S ? (Av)kf.dt : (Av)k.dt;

#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int v = 0; v < VC; ++v) {
      XF[q].v[v] = (H)first[q][0].v[v];
      XP[q].v[v] = (H)first[q][1].v[v];
      Y1F[q].v[v] = input(XF[q].v[v], dh, (Av)XP[q].v[v]);
    }
  const uint64_t t_begin = PACE ? __builtin_amdgcn_s_memrealtime() : 0;
  auto iteration = [&](auto phase, auto set, auto with_b, const int j) {
    // the value of plane P - d sits at [(phase - d) mod 3] of its history
    constexpr int p0 = decltype(phase)::value, p1 = (p0 + 2) % 3, p2 = (p0 + 1) % 3;
    constexpr int S = decltype(set)::value;  // j & 1: buffer set, prefetch slot
    H *bs = me + S * 4 * PL;
#pragma unroll
    for (int v = 0; v < VC; ++v) {
      XF[p0].v[v] = (H)LDF[S].v[v];
      XP[p0].v[v] = (H)LDP[S].v[v];
    }
    *(HV *)(bs) = XF[p1];
    *(HV *)(bs + PL) = Y1F[p1];
    *(HV *)(bs + 2 * PL) = Y2F[p2];
    *(HV *)(bs + 3 * PL) = Y3F[p2];
    load(S);  // plane P+2
    TbVec<float, VC> lf, lp;
    if constexpr (MODE != TB_F64) {
      lf = LF[S];
      lp = LP[S];
      load_lo(S, j + 2);
    }
    TbSite site_1[VC] = {}, site_2[VC] = {}, site_4[VC] = {};
#pragma unroll
    for (int v = 0; v < VC; ++v) {
      if constexpr (CURV) {
        site_1[v] = site_2[v] = tb_site<VAR>(psA[0].v[v], 0.0, k.m);
      } else if constexpr (COM || APX) {
        site_1[v] = tb_site<VAR>(psA[0].v[v], dpA[0].v[v], k.m);
        site_2[v] = tb_site<VAR>(psA[1].v[v], dpA[1].v[v], k.m);
        site_4[v] = tb_site<VAR>(psB.v[v], dpB.v[v], k.m);
      }
    }
    load_psi();
#pragma unroll
    for (int v = 0; v < VC; ++v) Y1F[p0].v[v] = input(XF[p0].v[v], dh, (Av)XP[p0].v[v]);
    if constexpr (PACE) {
      const uint64_t due = t_begin + (uint64_t)j * (uint64_t)u.pace;
      while (__builtin_amdgcn_s_memrealtime() < due) __builtin_amdgcn_s_sleep(1);
    }
    tb_barrier();

    // ---- A at P-1: k1 = f(x), k2 = f(y1)
    Av kp[VC];
    HV y1p, y2p;
    TbVec<Dv, VC> af, ap;
    force(XF[p1], XF[p0], XF[p2], XP[p1], bs, 0, site_1, kp);
#pragma unroll
    for (int v = 0; v < VC; ++v) {
      y1p.v[v] = input(XP[p1].v[v], dh, kp[v]);
      if constexpr (MODE == TB_F64) {
        af.v[v] = XF[p1].v[v] + k.dt6 * XP[p1].v[v];
        ap.v[v] = XP[p1].v[v] + k.dt6 * kp[v];
      } else {
        af.v[v] = (Dv)(k.dt6 * (double)XP[p1].v[v]);
        ap.v[v] = (Dv)(k.dt6 * (double)kp[v]);
      }
    }
    force(Y1F[p1], Y1F[p0], Y1F[p2], y1p, bs + PL, 1, site_2, kp);
#pragma unroll
    for (int v = 0; v < VC; ++v) {
      Y2F[p1].v[v] = input(XF[p1].v[v], dh, (Av)y1p.v[v]);
      y2p.v[v] = input(XP[p1].v[v], dh, kp[v]);
      af.v[v] = add(af.v[v], k.dt3, (double)y1p.v[v]);
      ap.v[v] = add(ap.v[v], k.dt3, (double)kp[v]);
      Y3F[p1].v[v] = input(XF[p1].v[v], dt, (Av)y2p.v[v]);
      af.v[v] = add(af.v[v], k.dt3, (double)y2p.v[v]);
    }
    // ---- B at P-2: k3 = f(y2), k4 = f(y3); new state (AF, AP, Y2P: from A of the
    // iteration before)
    if constexpr (decltype(with_b)::value != 0) {
      HV y3p;
      force(Y2F[p2], Y2F[p1], Y2F[p0], Y2P, bs + 2 * PL, 2, CURV || COM || APX ? site_mid : site_2, kp);
#pragma unroll
      for (int v = 0; v < VC; ++v) {
        y3p.v[v] = input(XP[p2].v[v], dt, kp[v]);
        AP.v[v] = add(AP.v[v], k.dt3, (double)kp[v]);
      }
      force(Y3F[p2], Y3F[p1], Y3F[p0], y3p, bs + 3 * PL, 3, CURV ? site_mid : site_4, kp);
      V of, op;
      if constexpr (MODE == TB_F64) {
#pragma unroll
        for (int v = 0; v < VC; ++v) {
          of.v[v] = AF.v[v] + k.dt6 * y3p.v[v];
          op.v[v] = AP.v[v] + k.dt6 * kp[v];
        }
      } else {
        TbVec<float, VC> olf, olp;
#pragma unroll
        for (int v = 0; v < VC; ++v) {
          double i0, i1;
          if constexpr (MODE == TB_F32S) {
            i0 = __builtin_fma(k.dt6, (double)y3p.v[v], AF.v[v]);
            i1 = __builtin_fma(k.dt6, (double)kp[v], AP.v[v]);
          } else {
            i0 = (double)AF.v[v] + k.dt6 * (double)y3p.v[v];
            i1 = (double)AP.v[v] + k.dt6 * kp[v];
          }
          const double s0 = ((double)XF[p2].v[v] + (double)lf.v[v]) + i0;
          const double s1 = ((double)XP[p2].v[v] + (double)lp.v[v]) + i1;
          of.v[v] = (float)s0;
          op.v[v] = (float)s1;
          olf.v[v] = (float)(s0 - (double)of.v[v]);
          olp.v[v] = (float)(s1 - (double)op.v[v]);
        }
        tb_store<float, VC>(olf, tb_plane(lout + off_st, plane_bytes), st_off);
        tb_store<float, VC>(olp, tb_plane(lout + N3 + off_st, plane_bytes), st_off);
      }
      tb_store<T, VC>(of, tb_plane(xout + off_st, plane_bytes), st_off);
      tb_store<T, VC>(op, tb_plane(xout + N3 + off_st, plane_bytes), st_off);
    }
    off_st = next_plane(off_st);
    Y2P = y2p;
    AF = af;
    AP = ap;
#pragma unroll
    for (int v = 0; v < VC; ++v) site_mid[v] = site_2[v];
  };
  iteration(tb_ic<2>{}, tb_ic<0>{}, tb_ic<0>{}, 2);
  iteration(tb_ic<0>{}, tb_ic<1>{}, tb_ic<0>{}, 3);
  for (int j = 4;;) {
    iteration(tb_ic<1>{}, tb_ic<0>{}, tb_ic<1>{}, j);
    if (++j >= iters) break;
    iteration(tb_ic<2>{}, tb_ic<1>{}, tb_ic<1>{}, j);
    if (++j >= iters) break;
    iteration(tb_ic<0>{}, tb_ic<0>{}, tb_ic<1>{}, j);
    if (++j >= iters) break;
    iteration(tb_ic<1>{}, tb_ic<1>{}, tb_ic<1>{}, j);
    if (++j >= iters) break;
    iteration(tb_ic<2>{}, tb_ic<0>{}, tb_ic<1>{}, j);
    if (++j >= iters) break;
    iteration(tb_ic<0>{}, tb_ic<1>{}, tb_ic<1>{}, j);
    if (++j >= iters) break;
  }
}

// Host: the step's scalars (runge_kutta4_classic.hpp:97-123 stage times; the
// RHS scalars as equations.cpp:75-80). inv_ah_sqr follows cf_inv_ah_sqr.
inline TbStep tb_step_host(const cf_kg_params *p, double t, double dt) {
  TbStep k;
  const double dh = dt / 2.0;
  const double th = t + dh;
  const double ts[4] = {t, th, th, t + dt};
  for (int s = 0; s < 4; ++s) {
    const double a_t = cf_cosmo_a(&p->cosmo, ts[s]);
    k.c_h[s] = (-3.0) * cf_cosmo_H(&p->cosmo, ts[s]);
    k.inv[s] = cf_inv_ah_sqr(p->N, p->L, a_t);
  }
  k.c_m = p->m * p->m;
  k.lam = p->lambda;
  k.m = p->m;
  k.fa2 = 0.0;
  k.dh = dh;
  k.dt = dt;
  k.dt6 = dt / 6.0;
  k.dt3 = dt / 3.0;
  return k;
}

}  // namespace cf
