// cf_adjoint.hip -- discrete adjoint of the RK4 lattice evolution and of the
// spectral loss  L = sum_s w_s P_rho(s)  (P_rho: the binned power spectrum of the
// energy density, compute_power_spectrum of fdm3d.cpp:7-34, at the final time).
//
// Loss adjoint. With rho_k the unnormalised DFT of rho and the bins summing the
// full k-cube, L = sum_k w_{s(k)} |rho_k|^2, so dL/drho(x) = 2 sum_k w rho_k e^{ikx}
// = 2 * C2R(w . rho_k): one D2Z, a per-mode multiply and one Z2D. The energy
// density (equations.cpp:106-138 with the lambda term of equations_cuda.cu:354)
//   rho = pi^2/2 + m^2 phi^2/2 + lambda phi^4/4 + (inv/8) sum_d (phi(x+e_d) - phi(x-e_d))^2
// gives
//   dL/dpi(x)  = g(x) pi(x)
//   dL/dphi(x) = g(x) (m^2 phi + lambda phi^3)
//              + (inv/4) sum_d [ g(x-e_d)(phi(x) - phi(x-2e_d)) - g(x+e_d)(phi(x+2e_d) - phi(x)) ]
//   dL/dm     += sum_x g(x) m phi(x)^2.
//
// Step adjoint. For x' = x + h/6 k1 + h/3 k2 + h/3 k3 + h/6 k4 with k_i = f(y_{i-1}),
// y0 = x, y1 = x + h/2 k1, y2 = x + h/2 k2, y3 = x + h k3 (runge_kutta4_classic.hpp:
// 87-138), and lambda' = dL/dx':
//   a4 = h/6 lambda';                 ybar3 = J(y3)^T a4
//   a3 = h/3 lambda' + h ybar3;       ybar2 = J(y2)^T a3
//   a2 = h/3 lambda' + h/2 ybar2;     ybar1 = J(y1)^T a2
//   a1 = h/6 lambda' + h/2 ybar1
//   lambda = lambda' + ybar3 + ybar2 + ybar1 + J(x)^T a1
//   dL/dm += sum_i (df/dm at y_{i-1}) . a_i,  df/dm = [0, -2 m phi]
// where f = [pi, -3H pi - m^2 phi - lambda phi^3 + inv Lap phi] and
//   (J^T a)_phi = (-m^2 - 3 lambda phi^2) a_pi + inv (sum_nbr a_pi - 6 a_pi)
//   (J^T a)_pi  = a_phi - 3H a_pi.
// The backward step is one kernel (k_adj_step) that marches tiles of columns along
// a, recomputes the stage states it needs from x on the fly with the forward stage
// arithmetic, in the forward kernels' operation order (same bits), and keeps the
// intermediate adjoint fields in LDS.
//
// Checkpointing: the forward pass keeps the state every `ckpt` steps (the last
// segment's states as they are made); the backward pass recomputes one segment of
// states at a time. Every state is written where it is kept (x0 is its own checkpoint) and
// the last step writes the gradient, so nothing is copied. Scalars (L, dL/dm) come from
// block partials summed on the device in a fixed order, so every result is bit-reproducible,
// and the call waits for the device once. (With copies of the states, the spectrum and the
// partials summed on the host: 1323 against 1159 us for 16 steps at N=128.)
#include <cmath>
#include <utility>

#include "cf_march.hpp"
#include "cf_tb_body.hpp"

namespace cf {

constexpr int ADJ_BLOCKS = 512;

// Fixed-order tree sum of one value per thread over a block of NT threads (tid =
// linear thread index; sm: NT doubles of LDS).
template <int NT>
__device__ __forceinline__ void block_partial(double v, double *part_slot, int tid, double *sm) {
  __syncthreads();  // sm may still be read by an earlier sum
  sm[tid] = v;
  __syncthreads();
  for (int s = NT / 2; s > 0; s >>= 1) {
    if (tid < s) sm[tid] += sm[tid + s];
    __syncthreads();
  }
  if (tid == 0) *part_slot = sm[0];
}

// Coefficients of one backward step from t: the forward right-hand side at t
// (stage 1) and at t + dt/2 (stages 2 and 3), -3H and inv_ah_sqr at t + dt (stage 4).
struct AdjStep {
  RhsCoef r1, r2;
  double ch4, inv4;
  double dh, dt, dt3, dt6;  // dt/2, dt, dt/3, dt/6
  double two_m;             // 2m
};

// The transposed Jacobian applied to a at a site, phi component:
// (-m^2 - 3 lambda phi_y^2) a_pi + inv (sum of the six neighbours' a_pi - 6 a_pi).
__device__ __forceinline__ double jt_phi(double c_m, double lam, double phi_y, double inv, double a0, double nb) {
  return (-c_m - 3.0 * lam * phi_y * phi_y) * a0 + inv * (nb - 6.0 * a0);
}

// Geometry of the backward step: output tiles of Tb x Tc columns (the region of a shape
// without a border of two on every side, or the whole extent of a smaller lattice) over
// chunks of A planes, one work unit each.
struct AdjGeom {
  int64_t N;
  int shape;     // index into adj_shapes
  int Tb, Tc;    // tile edges along b and c
  int ntb, ntc;  // tiles along b and c
  int A;         // planes per chunk
  int total;     // ntb * ntc * chunks
};

// Backward step, fused.
//
// Only phi of each stage state enters the transposed Jacobian, and only at the
// site, and phi of a stage state is local in the previous one:
//   y1.phi = x.phi + h/2 x.pi,  y2.phi = x.phi + h/2 y1.pi,  y3.phi = x.phi + h y2.pi
// with y1.pi = x.pi + h/2 f_pi(x) and y2.pi = x.pi + h/2 f_pi(y1): every y_s.phi at
// a site follows from x within distance 1 (the forward stage arithmetic, so the
// same bits as the stored stage states). Likewise, with ybar_s = J(y_s)^T a_{s+1},
// ybar.pi = a.phi - 3H a.pi is local and only ybar.phi has a stencil, so
//   a4 = h/6 lambda'                         (local)
//   ybar3 (at y3)                            phi: stencil of a4.pi
//   a3 = h/3 lambda' + h ybar3               pi: local
//   ybar2 (at y2)                            phi: stencil of a3.pi
//   a2 = h/3 lambda' + h/2 ybar2             at the site
//   ybar1.pi = a2.phi - 3H a2.pi,  a1.pi = h/6 lambda'.pi + h/2 ybar1.pi
// all within distance 1 of lambda' and x (half A). The rest needs the stencils of
// w = (a2.pi, a1.pi) (half B):
//   ybar1.phi (at y1): stencil of a2.pi;  J(x)^T a1: stencil of a1.pi
//   lambda = ((lambda' + ybar4) + ybar3 + ybar1).phi + (J(x)^T a1).phi, and the pi
//   half ((lambda' + ybar4 + ybar3) + ybar2 + ybar1).pi + (J(x)^T a1).pi
// (the order of the running sum s).
//
// The march is that of the blocked forward step (cf_tb_body.hpp): each thread owns two
// neighbouring columns of a row of the region, takes x and lambda' at plane P = a0 - 2 + j
// in iteration j (loaded two iterations ahead through buffer resources over one plane)
// and runs, side by side,
//   A at P-1 (x.phi, y1.phi, a4.pi, a3.pi at P-2..P): half A; w and the sum s stay in registers
//   B at P-2 (w at P-3..P-1): half B; writes lambda
// The in-plane neighbours come from six LDS plane buffers (the four of A at P-1, w of P-2),
// written together at the start of the iteration; with two sets of them one barrier per
// plane suffices. The first output needs A from j = 2 on, so planes 0 and 1 come straight
// from their loads and iterations 2 and 3 have no B. Results of region edges reach no
// stored site and no sum. s and w never reach HBM; the step reads x and lambda'
// (2 x 16 B/site, times the region/tile area ratio) and writes lambda (16 B/site).
//
// What bounds it: of the 1.7 us a plane of a 28 x 36 region takes, FP64 issue is 0.8 and
// LDS 0.65 (two wavefronts per SIMD in step with the barrier overlap them only in part).
// One column per thread (1024 threads, 128 VGPRs) took 32.1 us at N=128 against 27.9, 22 x
// 68 regions spill. Before, with 28 x 28 tiles that share 128-byte lines with their
// neighbours, one column per thread and half A masked per lane: 44 us.
//
// part: 4 ADJ_BLOCKS slots of which a block fills one with its dL/dm (all four stages) and
// block 0 clears those of blocks beyond the grid. lo must not overlap x or lp.
template <bool LAM, class SH>
__global__ __launch_bounds__(SH::NT) void k_adj_step(AdjGeom g, AdjStep k, const double *x, const double *lp,
                                                     double *lo, double *part) {
  constexpr int VC = SH::VC, RC = SH::RC, PL = SH::PLANE;
  typedef TbVec<double, VC> V;
  __shared__ __attribute__((aligned(16))) double lds[12 * PL + 2 * RC];
  const int N = (int)g.N;
  const int64_t NN = g.N * g.N, N3 = NN * g.N;
  const int plane_bytes = (int)(NN * 8);
  const int tid = (int)threadIdx.x, r = tid / SH::TPR, cc = (tid % SH::TPR) * VC;
  const double c_m = k.r1.c_m, lam = k.r1.lam;
  double *me = lds + RC + r * RC + cc;
  double dm = 0.0;
  for (int q = blockIdx.x; q < g.total; q += gridDim.x) {
    const int u = xcd_order(q, g.total);
    const int tc = u % g.ntc, rest = u / g.ntc, tb = rest % g.ntb, ac = rest / g.ntb;
    const int b0 = tb * g.Tb, c0 = tc * g.Tc;
    const int64_t a0 = (int64_t)ac * g.A, a1 = (a0 + g.A < g.N) ? a0 + g.A : g.N;
    int b = (b0 - TBH + r) % N, c = (c0 - TBH + cc) % N;
    if (b < 0) b += N;
    if (c < 0) c += N;
    const bool out = r >= TBH && r < TBH + g.Tb && b0 + (r - TBH) < N && cc >= TBH && cc < TBH + g.Tc &&
                     c0 + (cc - TBH) < N;
    const uint32_t ld_off = (uint32_t)(b * N + c) * 8u, st_off = out ? ld_off : TB_OOB;
    auto next_plane = [&](int64_t off) -> int64_t {
      off += NN;
      return off == N3 ? 0 : off;
    };
    int64_t off_ld = ((a0 - TBH) % g.N + g.N) % g.N * NN, off_st = off_ld;
    V LX[2], LXP[2], LL[2], LLP[2];
    auto load = [&](int s) {
      LX[s] = tb_load<double, VC>(tb_plane(x + off_ld, plane_bytes), ld_off);
      LXP[s] = tb_load<double, VC>(tb_plane(x + N3 + off_ld, plane_bytes), ld_off);
      LL[s] = tb_load<double, VC>(tb_plane(lp + off_ld, plane_bytes), ld_off);
      LLP[s] = tb_load<double, VC>(tb_plane(lp + N3 + off_ld, plane_bytes), ld_off);
      off_ld = next_plane(off_ld);
    };
    // histories: the value of plane P - d at [(phase - d) mod 3]
    V X[3], XP[3], Y1[3], F4[3], G3[3], LF[3], LP[3], W0[3] = {}, W1[3] = {}, SF = {}, SI = {}, D = {};
    auto take = [&](int h, int s) {
#pragma unroll
      for (int v = 0; v < VC; ++v) {
        const double xf = LX[s].v[v], xp = LXP[s].v[v], lf = LL[s].v[v], li = LLP[s].v[v];
        X[h].v[v] = xf;
        XP[h].v[v] = xp;
        LF[h].v[v] = lf;
        LP[h].v[v] = li;
        Y1[h].v[v] = xf + k.dh * xp;
        F4[h].v[v] = k.dt6 * li;                                                  // a4.pi
        G3[h].v[v] = k.dt3 * li + k.dt * (k.dt6 * lf + k.ch4 * F4[h].v[v]);       // a3.pi
      }
    };
    load(0);
    load(1);
    take(0, 0);
    load(0);
    take(1, 1);
    load(1);
    // the sum of a field's neighbours at column v; o its own plane, hi and lw those above
    // and below, p its own slot in the plane buffer
    struct Nb {
      V up, dn;
      double nx, pv;
    };
    auto in_plane = [&](const double *p) {
      Nb n;
      n.nx = p[VC];
      n.pv = p[-1];
      n.up = *(const V *)(p + RC);
      n.dn = *(const V *)(p - RC);
      return n;
    };
    auto cn = [&](const V &o, const Nb &n, int v) { return v + 1 < VC ? o.v[v + 1 < VC ? v + 1 : v] : n.nx; };
    auto cp = [&](const V &o, const Nb &n, int v) { return v > 0 ? o.v[v > 0 ? v - 1 : v] : n.pv; };
    auto iteration = [&](auto phase, auto set, auto with_b) {
      constexpr int p0 = decltype(phase)::value, p1 = (p0 + 2) % 3, p2 = (p0 + 1) % 3;
      constexpr int S = decltype(set)::value;
      double *bs = me + S * 6 * PL;
      take(p0, S);
      *(V *)(bs) = X[p1];
      *(V *)(bs + PL) = Y1[p1];
      *(V *)(bs + 2 * PL) = F4[p1];
      *(V *)(bs + 3 * PL) = G3[p1];
      if constexpr (decltype(with_b)::value != 0) {
        *(V *)(bs + 4 * PL) = W0[p2];
        *(V *)(bs + 5 * PL) = W1[p2];
      }
      load(S);  // plane P+2
      tb_barrier();
      // ---- A at P-1
      V y1pi, y2phi, y3phi, sf, si, d;
      {
        const Nb n = in_plane(bs);
#pragma unroll
        for (int v = 0; v < VC; ++v)
          y1pi.v[v] = XP[p1].v[v] + k.dh * rhs_pi(X[p1].v[v], X[p0].v[v], X[p2].v[v], n.up.v[v], n.dn.v[v],
                                                  cn(X[p1], n, v), cp(X[p1], n, v), XP[p1].v[v], k.r1, LAM);
      }
      {
        const Nb n = in_plane(bs + PL);
#pragma unroll
        for (int v = 0; v < VC; ++v) {
          const double y2pi = XP[p1].v[v] + k.dh * rhs_pi(Y1[p1].v[v], Y1[p0].v[v], Y1[p2].v[v], n.up.v[v],
                                                          n.dn.v[v], cn(Y1[p1], n, v), cp(Y1[p1], n, v), y1pi.v[v],
                                                          k.r2, LAM);
          y2phi.v[v] = X[p1].v[v] + k.dh * y1pi.v[v];
          y3phi.v[v] = X[p1].v[v] + k.dt * y2pi;
        }
      }
      V yb4phi;
      {  // stage 4 at y3 (t + dt)
        const Nb n = in_plane(bs + 2 * PL);
#pragma unroll
        for (int v = 0; v < VC; ++v) {
          const double nb = F4[p0].v[v] + F4[p2].v[v] + n.up.v[v] + n.dn.v[v] + cn(F4[p1], n, v) + cp(F4[p1], n, v);
          yb4phi.v[v] = jt_phi(c_m, lam, y3phi.v[v], k.inv4, F4[p1].v[v], nb);
        }
      }
      {  // stage 3 at y2 and the local part of stage 2 at y1 (t + dt/2)
        const Nb n = in_plane(bs + 3 * PL);
#pragma unroll
        for (int v = 0; v < VC; ++v) {
          const double fc = F4[p1].v[v], gc = G3[p1].v[v], lf = LF[p1].v[v], li = LP[p1].v[v];
          const double nb = G3[p0].v[v] + G3[p2].v[v] + n.up.v[v] + n.dn.v[v] + cn(G3[p1], n, v) + cp(G3[p1], n, v);
          const double yb3phi = jt_phi(c_m, lam, y2phi.v[v], k.r2.inv, gc, nb);
          const double yb4pi = k.dt6 * lf + k.ch4 * fc;
          const double yb3pi = (k.dt3 * lf + k.dt * yb4phi.v[v]) + k.r2.c_h * gc;
          const double a2pi = k.dt3 * li + k.dh * yb3pi;
          const double a2phi = k.dt3 * lf + k.dh * yb3phi;
          const double yb2pi = a2phi + k.r2.c_h * a2pi;
          d.v[v] = y3phi.v[v] * fc + y2phi.v[v] * gc + Y1[p1].v[v] * a2pi;
          sf.v[v] = (lf + yb4phi.v[v]) + yb3phi;
          si.v[v] = ((li + yb4pi) + yb3pi) + yb2pi;
          W0[p1].v[v] = a2pi;
          W1[p1].v[v] = k.dt6 * li + k.dh * yb2pi;
        }
      }
      // ---- B at P-2 (SF, SI, D: from A of the iteration before)
      if constexpr (decltype(with_b)::value != 0) {
        const Nb nu = in_plane(bs + 4 * PL), nv = in_plane(bs + 5 * PL);
        V of, op;
#pragma unroll
        for (int v = 0; v < VC; ++v) {
          const double xf = X[p2].v[v], um1 = W0[p2].v[v], vm1 = W1[p2].v[v];
          const double nb2 = W0[p1].v[v] + W0[p0].v[v] + nu.up.v[v] + nu.dn.v[v] + cn(W0[p2], nu, v) + cp(W0[p2], nu, v);
          const double yb2phi = jt_phi(c_m, lam, Y1[p2].v[v], k.r2.inv, um1, nb2);
          const double nb1 = W1[p1].v[v] + W1[p0].v[v] + nv.up.v[v] + nv.dn.v[v] + cn(W1[p2], nv, v) + cp(W1[p2], nv, v);
          const double outphi = jt_phi(c_m, lam, xf, k.r1.inv, vm1, nb1);
          const double outpi = (k.dt6 * LF[p2].v[v] + k.dh * yb2phi) + k.r1.c_h * vm1;
          of.v[v] = (SF.v[v] + yb2phi) + outphi;
          op.v[v] = SI.v[v] + outpi;
          const double s = D.v[v] + xf * vm1;
          dm += out ? -k.two_m * s : 0.0;
        }
        tb_store<double, VC>(of, tb_plane(lo + off_st, plane_bytes), st_off);
        tb_store<double, VC>(op, tb_plane(lo + N3 + off_st, plane_bytes), st_off);
      }
      off_st = next_plane(off_st);
      SF = sf;
      SI = si;
      D = d;
    };
    const int iters = (int)(a1 - a0) + 4;
    iteration(tb_ic<2>{}, tb_ic<0>{}, tb_ic<0>{});
    iteration(tb_ic<0>{}, tb_ic<1>{}, tb_ic<0>{});
    for (int j = 4;;) {
      iteration(tb_ic<1>{}, tb_ic<0>{}, tb_ic<1>{});
      if (++j >= iters) break;
      iteration(tb_ic<2>{}, tb_ic<1>{}, tb_ic<1>{});
      if (++j >= iters) break;
      iteration(tb_ic<0>{}, tb_ic<0>{}, tb_ic<1>{});
      if (++j >= iters) break;
      iteration(tb_ic<1>{}, tb_ic<1>{}, tb_ic<1>{});
      if (++j >= iters) break;
      iteration(tb_ic<2>{}, tb_ic<0>{}, tb_ic<1>{});
      if (++j >= iters) break;
      iteration(tb_ic<0>{}, tb_ic<1>{}, tb_ic<1>{});
      if (++j >= iters) break;
    }
    tb_barrier();  // the plane buffers are read until here: the next unit, or the sum below
  }
  // fixed-order sum over the block: within the wavefronts, then over them
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) dm += __shfl_xor(dm, s);
  if ((tid & 63) == 0) lds[tid >> 6] = dm;
  __syncthreads();
  if (tid == 0) {
    double t = 0.0;
    for (int w = 0; w < SH::NT / 64; ++w) t += lds[w];
    part[blockIdx.x] = t;
  }
  if (blockIdx.x == 0)
    for (int sl = (int)gridDim.x + tid; sl < 4 * ADJ_BLOCKS; sl += SH::NT) part[sl] = 0.0;
}

// Region shapes of the backward step, smallest first: blocks that a CU holds at a time (the
// two-column kernels take 230-245 VGPRs, two wavefronts per SIMD), the time of a plane
// iteration in us with one block on the CU and, per block, with all of them.
typedef TbShape<12, 20, 2, 128> AdjS12x20;
typedef TbShape<14, 36, 1, 512> AdjS14x36;
typedef TbShape<28, 36, 2, 512> AdjS28x36;
struct AdjShapeInfo {
  int rb, rc, resident;
  double t1, tau;
};

// Shape and chunk of the backward step: the least modelled time, the larger of the busiest
// CU's plane iterations (chunk + 2 each, as in tb_cost) and the bytes passed at 5.5 TB/s
// (8.8 while they fit the 256 MB cache). Measured (us a step; one rule over 32 x 32 regions
// of 28 x 28 tiles / here; the same N with the other shapes): N=32 14 / 5.6 (6.1, 7.6),
// 64 23 / 8.8 (10.5, 10.0), 128 44 / 27.9 (32.6, 30.6), 256 290 / 200 (-, 225).
static AdjGeom adj_geom(int64_t N) {
  static const AdjShapeInfo shapes[3] = {
      {12, 20, 4, 0.80, 0.43}, {14, 36, 1, 0.87, 0.87}, {28, 36, 1, 1.75, 1.75}};
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
    cus = 256;
  AdjGeom best{};
  double best_cost = -1.0;
  for (int s = 0; s < 3; ++s) {
    const AdjShapeInfo &sh = shapes[s];
    AdjGeom g;
    g.N = N;
    g.shape = s;
    g.Tb = N < sh.rb - 2 * TBH ? (int)N : sh.rb - 2 * TBH;
    g.Tc = N < sh.rc - 2 * TBH ? (int)N : sh.rc - 2 * TBH;
    g.ntb = (int)cdiv(N, g.Tb);
    g.ntc = (int)cdiv(N, g.Tc);
    for (int64_t k = 1; k <= N;) {  // every distinct ceil(N / k)
      g.A = (int)cdiv(N, k);
      g.total = g.ntb * g.ntc * (int)cdiv(N, g.A);
      const int64_t n = cdiv(g.total, cus), full = n / sh.resident, rest = n % sh.resident;
      const double one = std::max(sh.t1, (double)rest * sh.tau);
      const double cu = 3.2 + (double)(g.A + 2) * ((double)full * sh.resident * sh.tau + (rest ? one : 0.0));
      const double loads = 32.0 * (double)g.total * sh.rb * sh.rc * (double)(g.A + 2 * TBH);
      const double sites = (double)N * (double)N * (double)N;
      const double bw = 48.0 * sites <= 256e6 ? 8.8e6 : 5.5e6;
      const double cost = std::max(cu, (loads + 16.0 * sites) / bw);
      if (best_cost < 0.0 || cost < best_cost) {
        best = g;
        best_cost = cost;
      }
      k = g.A > 1 ? (N + g.A - 2) / (g.A - 1) : N + 1;
    }
  }
  return best;
}

template <bool LAM>
static void adj_launch(const AdjGeom &g, const AdjStep &k, const double *x, const double *li, double *lo, double *part,
                       hipStream_t st) {
  const dim3 grid(g.total < 4 * ADJ_BLOCKS ? g.total : 4 * ADJ_BLOCKS);
  if (g.shape == 0)
    hipLaunchKernelGGL((k_adj_step<LAM, AdjS12x20>), grid, dim3(AdjS12x20::NT), 0, st, g, k, x, li, lo, part);
  else if (g.shape == 1)
    hipLaunchKernelGGL((k_adj_step<LAM, AdjS14x36>), grid, dim3(AdjS14x36::NT), 0, st, g, k, x, li, lo, part);
  else
    hipLaunchKernelGGL((k_adj_step<LAM, AdjS28x36>), grid, dim3(AdjS28x36::NT), 0, st, g, k, x, li, lo, part);
}

// Energy-density adjoint: g (N^3) -> gx (2N^3); part[block] = sum g m phi^2. A thread owns
// two neighbouring columns of a chunk of planes, as in the energy density (cf_stencil.hip);
// blocks walk over the tiles. N=128: 18.7 us (one site per thread and pass, its fifteen
// neighbours by 64-bit division: 31).
constexpr int RA_TC = 64, RA_TB = 4, RA_A = 8;  // column pairs, rows and planes of a tile
__global__ __launch_bounds__(RA_TC *RA_TB) void k_rho_adjoint(int64_t N64, int nct, int nbt, int total,
                                                              const double *__restrict__ x,
                                                              const double *__restrict__ g, double *__restrict__ gx,
                                                              double m, double lam, double inv,
                                                              double *__restrict__ part) {
  typedef TbVec<double, 2> V;
  __shared__ double sm[RA_TC * RA_TB];
  const int N = (int)N64, bytes = (int)(N64 * N64 * 8);
  const int64_t NN = N64 * N64, N3 = NN * N64;
  const double q = 0.25 * inv, mm = m * m;
  double dm = 0.0;
  for (int block = xcd_order((int)blockIdx.x, (int)gridDim.x); block < total; block += (int)gridDim.x) {
    const int ct = block % nct, rest = block / nct, bt = rest % nbt, a0 = rest / nbt * RA_A;
    const int c = 2 * (ct * RA_TC + (int)(threadIdx.x & (RA_TC - 1))), b = bt * RA_TB + (int)(threadIdx.x / RA_TC);
    if (c >= N || b >= N) continue;
    const int a1 = a0 + RA_A < N ? a0 + RA_A : N;
    auto wrap = [&](int i) { return i < 0 ? i + N : (i >= N ? i - N : i); };
    auto off = [&](int bb, int cc) { return (uint32_t)(wrap(bb) * N + wrap(cc)) * 8u; };
    const uint32_t own = off(b, c);
    const uint32_t xb2 = off(b + 2, c), xb_2 = off(b - 2, c), gb1 = off(b + 1, c), gb_1 = off(b - 1, c);
    const uint32_t xc2 = off(b, c + 2), xc_2 = off(b, c - 2), gc2 = off(b, c + 2), gc_1 = off(b, c - 1);
    auto xp = [&](int a) { return tb_plane(x + (int64_t)wrap(a) * NN, bytes); };
    auto gp = [&](int a) { return tb_plane(g + (int64_t)wrap(a) * NN, bytes); };
    auto ld = [&](__amdgpu_buffer_rsrc_t r, uint32_t o) { return tb_load<double, 2>(r, o); };
    V x_2 = ld(xp(a0 - 2), own), x_1 = ld(xp(a0 - 1), own), x0 = ld(xp(a0), own), x1 = ld(xp(a0 + 1), own);
    V g_1 = ld(gp(a0 - 1), own), g0 = ld(gp(a0), own);
#pragma unroll 2
    for (int a = a0; a < a1; ++a) {
      const auto rx = xp(a), rg = gp(a);
      const V x2 = ld(xp(a + 2), own), g1 = ld(gp(a + 1), own);
      const V ub = ld(rx, xb2), db = ld(rx, xb_2), ugb = ld(rg, gb1), dgb = ld(rg, gb_1);
      const V uc = ld(rx, xc2), dc = ld(rx, xc_2);
      const double gr = tb_load<double, 1>(rg, gc2).v[0], gl = tb_load<double, 1>(rg, gc_1).v[0];
      const V pi = ld(tb_plane(x + N3 + (int64_t)a * NN, bytes), own);
      V of, op;
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        const double phi = x0.v[v], gs = g0.v[v];
        double gphi = gs * (mm * phi + lam * phi * phi * phi);
        gphi += q * (g_1.v[v] * (phi - x_2.v[v]) - g1.v[v] * (x2.v[v] - phi));
        gphi += q * (dgb.v[v] * (phi - db.v[v]) - ugb.v[v] * (ub.v[v] - phi));
        const double gm = v == 0 ? gl : g0.v[0], gq = v == 0 ? g0.v[1] : gr;
        gphi += q * (gm * (phi - dc.v[v]) - gq * (uc.v[v] - phi));
        of.v[v] = gphi;
        op.v[v] = gs * pi.v[v];
        dm += gs * m * phi * phi;
      }
      tb_store<double, 2>(of, tb_plane(gx + (int64_t)a * NN, bytes), own);
      tb_store<double, 2>(op, tb_plane(gx + N3 + (int64_t)a * NN, bytes), own);
      x_2 = x_1;
      x_1 = x0;
      x0 = x1;
      x1 = x2;
      g_1 = g0;
      g0 = g1;
    }
  }
  block_partial<RA_TC * RA_TB>(dm, part + blockIdx.x, (int)threadIdx.x, sm);
}

// One block: *out = sum of a (times b where given), in a fixed order.
__global__ __launch_bounds__(1024) void k_sum(const double *__restrict__ a, const double *__restrict__ b, int64_t n,
                                              double *__restrict__ out) {
  __shared__ double sm[1024];
  double s = 0.0;
#pragma unroll 8
  for (int64_t i = threadIdx.x; i < n; i += 1024) s += b ? a[i] * b[i] : a[i];
  block_partial<1024>(s, out, (int)threadIdx.x, sm);
}

// Launches of cf_loss_spectrum_adjoint; res (device) <- L, dL/dm.
static cf_status loss_adjoint(cf_spectrum_plan *plan, const cf_kg_params *p, const double *x, double t,
                              const double *weights, double *gx, double *scratch, double *res, hipStream_t st) {
  const int64_t N = p->N, nb = cf_spectrum_bins(N);
  const double inv = cf_inv_ah_sqr(N, p->L, cf_cosmo_a(&p->cosmo, t));
  double *rho = scratch;
  CF_TRY(cf_energy_density_f64(N, x, rho, p->m, p->lambda, inv, st));
  double *fk = gx;  // the half spectrum (2 N^2 H doubles) fits in gx (2N^3) until rho's gradient is formed
  CF_TRY(cf_fft_d2z(plan, rho, fk, st));
  double *bins = plan_bins(plan), *part = plan_red(plan);
  CF_TRY(cf_bin_power(plan, fk, bins, st));
  hipLaunchKernelGGL(k_sum, dim3(1), dim3(1024), 0, st, bins, weights, nb, res);
  CF_LAUNCHED();
  CF_TRY(plan_z2d_weighted(plan, fk, weights, rho, st));  // rho <- dL/drho
  const int nct = (int)cdiv(N / 2, RA_TC), nbt = (int)cdiv(N, RA_TB), total = nct * nbt * (int)cdiv(N, RA_A);
  const int blocks = total < 2 * ADJ_BLOCKS ? total : 2 * ADJ_BLOCKS;
  static_assert(2 * ADJ_BLOCKS <= 1025, "dL/dm partials live in the plan's reduction buffer");
  hipLaunchKernelGGL(k_rho_adjoint, dim3(blocks), dim3(RA_TC * RA_TB), 0, st, N, nct, nbt, total, x, rho, gx, p->m,
                     p->lambda, inv, part);
  CF_LAUNCHED();
  hipLaunchKernelGGL(k_sum, dim3(1), dim3(1024), 0, st, part, nullptr, (int64_t)blocks, res + 1);
  CF_LAUNCHED();
  return CF_OK;
}

}  // namespace cf

using namespace cf;

extern "C" {

size_t cf_adjoint_work_bytes(int64_t N, int64_t n_steps, int64_t ckpt) {
  if (!valid_N(N) || n_steps < 0 || ckpt <= 0) return 0;
  const size_t v = 2 * (size_t)N * N * N * sizeof(double);
  const size_t nck = (size_t)((n_steps + ckpt - 1) / ckpt);
  // checkpoints + one segment of states + lambda (2) + forward work (3). Callers size buffers
  // by this; of it the first and last checkpoint (x0 itself; kept with the last segment) and
  // the third work vector are not touched.
  return nck * v + (size_t)ckpt * v + 2 * v + 3 * v +
         (size_t)(4 * n_steps + 1) * ADJ_BLOCKS * sizeof(double);
}

// L and dL/dx (gx_dev, 2N^3) and the direct dL/dm at a state x; weights_dev has
// cf_spectrum_bins(N) entries. scratch_dev: N^3 doubles. Blocking (L, dL/dm on host).
cf_status cf_loss_spectrum_adjoint(cf_spectrum_plan *plan, const cf_kg_params *p, const double *x, double t,
                                   const double *weights_dev, double *gx_dev, double *scratch_dev, double *loss,
                                   double *dldm, cf_stream stream) {
  CF_REQUIRE(plan && p && x && weights_dev && gx_dev && scratch_dev && loss && dldm,
             "cf_loss_spectrum_adjoint: null argument");
  CF_REQUIRE(plan_size(plan) == p->N, "cf_loss_spectrum_adjoint: plan is for N=%lld, lattice N=%lld",
             (long long)plan_size(plan), (long long)p->N);
  hipStream_t st = S(stream);
  double *res = plan_bins(plan) + cf_spectrum_bins(p->N), host[2];
  CF_TRY(loss_adjoint(plan, p, x, t, weights_dev, gx_dev, scratch_dev, res, st));
  CF_HIP(hipMemcpyAsync(host, res, sizeof(host), hipMemcpyDeviceToHost, st));
  CF_HIP(hipStreamSynchronize(st));
  *loss = host[0];
  *dldm = host[1];
  return CF_OK;
}

// One backward step from state x at time t: lo = dL/dx_n from li = dL/dx_{n+1};
// part: 4*ADJ_BLOCKS partials of dL/dm, one per block over all four stages, zero beyond the
// grid. lo overlaps neither x nor li.
static cf_status adj_step(const cf_kg_params *p, const double *x, double t, double dt, const double *li, double *lo,
                          double *part, hipStream_t st) {
  const int64_t N = p->N;
  const double dh = dt / 2.0, th = t + dh;
  auto rhs = [&](double tt) {
    RhsCoef r;
    r.c_h = (-3.0) * cf_cosmo_H(&p->cosmo, tt);
    r.c_m = p->m * p->m;
    r.lam = p->lambda;
    r.inv = cf_inv_ah_sqr(N, p->L, cf_cosmo_a(&p->cosmo, tt));
    return r;
  };
  AdjStep k;
  k.r1 = rhs(t);
  k.r2 = rhs(th);
  const RhsCoef r4 = rhs(t + dt);
  k.ch4 = r4.c_h;
  k.inv4 = r4.inv;
  k.dh = dh;
  k.dt = dt;
  k.dt3 = dt / 3.0;
  k.dt6 = dt / 6.0;
  k.two_m = 2.0 * p->m;
  const AdjGeom g = adj_geom(N);
  if (p->lambda != 0.0) adj_launch<true>(g, k, x, li, lo, part, st);
  else adj_launch<false>(g, k, x, li, lo, part, st);
  CF_LAUNCHED();
  return CF_OK;
}

// One RK4 step adjoint at state x_n (time t): lam_dev holds dL/dx_{n+1} on entry and
// dL/dx_n on return; the step's dL/dm contributions go to part_dev (4*ADJ_BLOCKS
// doubles, summed by the caller). work_dev: 2N^3 doubles.
cf_status cf_rk4_step_adjoint_f64(const cf_kg_params *p, const double *x, double t, double dt, double *lam,
                                  double *part_dev, void *work_dev, cf_stream stream) {
  CF_REQUIRE(p && x && lam && part_dev && work_dev, "cf_rk4_step_adjoint_f64: null argument");
  CF_REQUIRE(valid_N(p->N), "cf_rk4_step_adjoint_f64: unsupported N");
  const int64_t N = p->N, n = 2 * N * N * N;
  hipStream_t st = S(stream);
  double *lo = (double *)work_dev;
  CF_TRY(adj_step(p, x, t, dt, lam, lo, part_dev, st));
  CF_HIP(hipMemcpyAsync(lam, lo, n * sizeof(double), hipMemcpyDeviceToDevice, st));
  return CF_OK;
}

// Forward n_steps from x0 (t_k = t0 + k dt) with checkpoints every ckpt steps, the
// spectral loss at t_end, and the backward pass: grad_x0_dev = dL/dx0 (2N^3),
// *loss = L, *dldm = dL/dm (direct loss term + every step). Blocking.
cf_status cf_adjoint_spectrum_loss(cf_spectrum_plan *plan, const cf_kg_params *p, const double *x0, double t0,
                                   double dt, int64_t n_steps, int64_t ckpt, const double *weights_dev,
                                   double *grad_x0_dev, double *loss, double *dldm, void *work_dev,
                                   cf_stream stream) {
  CF_REQUIRE(plan && p && x0 && weights_dev && grad_x0_dev && loss && dldm && work_dev && n_steps >= 0 && ckpt > 0,
             "cf_adjoint_spectrum_loss: bad arguments");
  CF_REQUIRE(valid_N(p->N), "cf_adjoint_spectrum_loss: unsupported N");
  CF_REQUIRE(plan_size(plan) == p->N, "cf_adjoint_spectrum_loss: plan is for N=%lld, lattice N=%lld",
             (long long)plan_size(plan), (long long)p->N);
  const int64_t N = p->N, n = 2 * N * N * N;
  const size_t vb = (size_t)n * sizeof(double);
  hipStream_t st = S(stream);
  const int64_t nck = (n_steps + ckpt - 1) / ckpt;
  double *ck = (double *)work_dev;                // nck checkpoints
  double *seg = ck + (size_t)nck * n;              // ckpt states of one segment
  double *lamb = seg + (size_t)ckpt * n;           // lambda, two buffers taken in turn
  double *lamb2 = lamb + n;
  double *fw = lamb2 + n;                          // forward work: 3 vectors
  double *part = fw + 3 * n;                       // 4 n_steps * ADJ_BLOCKS
  double *res = plan_bins(plan) + cf_spectrum_bins(N);  // L, dL/dm of the loss and of the steps
  auto step = [&](int64_t k, const double *from, double *to) {  // same bits as the stage kernels
    return cf_rk4_step_tb_f64(p, from, to, t0 + static_cast<double>(k) * dt, dt, 0, stream);
  };
  // Start of a segment: x0 itself, or its checkpoint; the last one's states are all kept in
  // seg as they are made, its start there too, so the backward pass does not recompute them.
  auto start = [&](int64_t c) -> const double * {
    return c == 0 ? x0 : (c + 1 == nck ? seg : ck + (size_t)c * n);
  };
  auto state = [&](int64_t c, int64_t k) -> const double * {  // state k of segment c, once in seg
    return k == c * ckpt ? start(c) : seg + (size_t)(k - c * ckpt) * n;
  };
  // forward: every step into the buffer that keeps its result, the others in turn into two
  // work vectors; the final state into lamb2, which the loss adjoint leaves alone and the
  // backward pass overwrites only after the loss
  const double *x = x0;
  for (int64_t k = 0; k < n_steps; ++k) {
    const int64_t c = k / ckpt, next = k + 1;
    double *to = next == n_steps    ? lamb2
                 : c + 1 == nck     ? seg + (size_t)(next - c * ckpt) * n
                 : next % ckpt == 0 ? const_cast<double *>(start(c + 1))
                                    : fw + (size_t)(next & 1) * n;
    CF_TRY(step(k, x, to));
    x = to;
  }
  const double t_end = t0 + static_cast<double>(n_steps) * dt;
  CF_TRY(loss_adjoint(plan, p, x, t_end, weights_dev, lamb, fw, res, st));
  // backward, one segment at a time; the last step writes the gradient (through lamb2 where
  // it shares memory with x0, which that step reads)
  const char *gb = (const char *)grad_x0_dev, *xb = (const char *)x0;
  const bool direct = gb + vb <= xb || xb + vb <= gb;
  for (int64_t c = nck - 1; c >= 0; --c) {
    const int64_t k0 = c * ckpt, k1 = (k0 + ckpt < n_steps) ? k0 + ckpt : n_steps;
    for (int64_t k = k0; k + 1 < k1 && c + 1 < nck; ++k)
      CF_TRY(step(k, state(c, k), seg + (size_t)(k + 1 - k0) * n));
    for (int64_t k = k1 - 1; k >= k0; --k) {
      const double t = t0 + static_cast<double>(k) * dt;
      double *to = k == 0 && direct ? grad_x0_dev : lamb2;
      CF_TRY(adj_step(p, state(c, k), t, dt, lamb, to, part + (size_t)k * 4 * ADJ_BLOCKS, st));
      std::swap(lamb, lamb2);
      if (to == grad_x0_dev) lamb = grad_x0_dev;
    }
  }
  hipLaunchKernelGGL(k_sum, dim3(1), dim3(1024), 0, st, part, nullptr, n_steps * 4 * ADJ_BLOCKS, res + 2);
  CF_LAUNCHED();
  double host[3];
  if (lamb != grad_x0_dev) CF_HIP(hipMemcpyAsync(grad_x0_dev, lamb, vb, hipMemcpyDeviceToDevice, st));
  CF_HIP(hipMemcpyAsync(host, res, sizeof(host), hipMemcpyDeviceToHost, st));
  CF_HIP(hipStreamSynchronize(st));
  *loss = host[0];
  *dldm = host[1] + host[2];
  return CF_OK;
}

}  // extern "C"
