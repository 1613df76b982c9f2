// swm_kernels.hip -- FP64 HIP kernels (gfx950) of the WENO5 time steps of
// sw-mpdec -- mPDeC5 and the other modified-Patankar schemes of the PATANKAR
// build, and the explicit schemes of the build without it -- over all active
// jobs of an engine.
//
// One FVTimeDerivative (src/finitevolume.f90:402-440) covers every job and up
// to three DeC nodes:
//   k_fvtd         x faces: halo tile -> ConsToPrim -> WENO5 first sweep along
//                  x (shared through LDS) -> second sweep along y at the 4 Gauss
//                  points -> positivity limiter on h -> Rusanov -> Gauss sum;
//                  y faces: the same; source term (h-only WENO5 point values
//                  times -g db): one launch where the device would be left
//                  idle, launches of their own on large grids
//   the update     UpdateTimeDerivative: Ut(2:3) and face mass fluxes / dx, in
//                  k_fvtd_update, with the sources in k_fvtd_source_update, or
//                  inside the assembly that reads them
// The Patankar assembly carries the DeC momentum update of the same nodes
// (disjoint arrays).  k_solve runs the Jacobi iteration of the grids whose
// systems fit the register files, stop decisions included (swm_engine.cpp,
// solve_tables).  Larger grids get a launch per sweep: the first inside the
// assembly, each with per-block sums of |x_new - x_old|, and a one-block-per-job
// kernel takes the stop decision of src/jacobi_iteration.f90:71 on the device.
// Outside k_solve no grid-wide waits are used: on a multi-XCD device an
// agent-scope fence writes back the L2, so the kernel boundary is the cheap way
// to publish partial sums.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "swm_engine.hpp"
#include "swm_numerics.hpp"
#include "swm_timestep.hpp"

namespace swm {

// thetaDeC: THETA[b][m][r] = thetaDeC(m+1, r+1) of block b
//   b = 0  mPDeC5  (src/timediscretization.f90:491-506)
//   b = 1  mPEuler and mPDeC2, reshape((/0, 1/2, 0, 1/2/), (/2,2/))
//          (src/timediscretization.f90:604,704)
#define SWM_THETA_TABLE                                                                         \
  {{{0.0000000000000000000, 0.0000000000000000000, 0.0000000000000000000, 0.0000000000000000000},  \
    {0.1103005664791649049, 0.1896994335208351257, -0.0339073642291439076, 0.0103005664791649201}, \
    {0.0730327668541684294, 0.4505740308958107176, 0.2269672331458314485, -0.0269672331458315692}, \
    {0.0833333333333333287, 0.4166666666666666852, 0.4166666666666666852, 0.0833333333333333287}}, \
   {{0.0, 0.0, 0.0, 0.0}, {0.5, 0.5, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}}}
__constant__ double THETA[2][4][4] = SWM_THETA_TABLE;

// Sign pattern of THETA[b][m][.]: bit r set when thetaDeC(m+1, r+1) > 0.  The
// assembly branches on it, uniformly for a whole launch.
constexpr double kThetaHost[2][4][4] = SWM_THETA_TABLE;
constexpr int theta_pos(int b, int m) {
  int p = 0;
  for (int r = 0; r < 4; ++r)
    if (kThetaHost[b][m][r] > 0.) p |= 1 << r;
  return p;
}
__constant__ int THETA_POS[2][4] = {{theta_pos(0, 0), theta_pos(0, 1), theta_pos(0, 2), theta_pos(0, 3)},
                                    {theta_pos(1, 0), theta_pos(1, 1), theta_pos(1, 2), theta_pos(1, 3)}};
static_assert(theta_pos(0, 1) == 0xB && theta_pos(0, 2) == 0x7 && theta_pos(0, 3) == 0xF &&
                  theta_pos(1, 1) == 0x3,
              "thetaDeC sign pattern");

// Global-address-space view of a device array.  The arrays' pointers are read
// from the job table in memory, so the compiler cannot infer their address
// space and would use flat loads and stores, which also occupy the LDS wait
// counter; through G() they become global loads and stores.
typedef __attribute__((address_space(1))) double gdouble;
__device__ __forceinline__ const gdouble* G(const double* p) { return (const gdouble*)p; }
__device__ __forceinline__ gdouble* G(double* p) { return (gdouble*)p; }

// 0-based index of Fortran cell c (1..n or a periodic ghost) on an axis of n.
// The tiles' halos keep c within [-2, n + 17], so one add or subtract of n
// suffices for n >= 17; smaller axes take the modulo.
__device__ __forceinline__ int wrap1(int c, int n) {
  int m = c - 1;
  if (m < 0)
    m += n;
  else if (m >= n)
    m -= n;
  if ((unsigned)m >= (unsigned)n) {
    m = (c - 1) % n;
    if (m < 0) m += n;
  }
  return m;
}

// Row-major cell k = k0 + t of a grid nx wide, with (i0, j0) the cell of k0
// (computed once per block): i = k % nx, j = k / nx without a per-thread
// integer division.
__device__ __forceinline__ void cell_ij(int i0, int j0, int t, int nx, int& i, int& j) {
  i = i0 + t;
  j = j0;
  while (i >= nx) {
    i -= nx;
    ++j;
  }
}

// v of the lane that CTRL of the DPP encoding names; 0 where there is none, and
// in the rows of 16 lanes left out of ROWS.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, true);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ int cdiv_d(int a, int b) { return (a + b - 1) / b; }

// In the steps of a batch (E.gated) a job whose batch has stopped
// (JobStatus::halt) is skipped by every kernel; the test is uniform per block.
// The status is reached from the launch's arguments, not through the job's
// descriptor: a small kernel is a chain of dependent loads of 0.5 to 1 us each
// (arguments, block's tile, job's descriptor, its data), and the look-ups saved
// here and in tile_of and job_of are most of what its latency can lose.
__device__ __forceinline__ bool skipped(const EngineArgs& E, int job) {
  return E.gated && E.status[job].halt != 0;
}

// The same for kernels that write only stage buffers, which the next step
// computes anew: one small grid is not worth the load (halt was written by
// another XCD, so it comes from memory before anything else may start; 1 us of
// a kernel of 4 to 5), its steps after a stop run in vain, uncommitted.
__device__ __forceinline__ bool skipped_stage(const EngineArgs& E, int job) {
  return E.gated && !E.eager && E.status[job].halt != 0;
}

// Entry b of a table of tiles or of jobs.
__device__ __forceinline__ TileRef tile_of(const EngineArgs& E, const TileRef* tiles, int b) {
  if (E.single >= 0) return {E.single, b};
  return tiles[b];
}
__device__ __forceinline__ int job_of(const EngineArgs& E, const int* jobs, int b) {
  return E.single >= 0 ? E.single : jobs[b];
}

// State slot m of a job: m = 0 is U^n, 1..3 the DeC nodes.
__device__ __forceinline__ void node_state(const JobDev& J, int m, const gdouble*& h,
                                           const gdouble*& hu, const gdouble*& hv) {
  h = G(J.sh[m]);
  hu = G(J.shu[m]);
  hv = G(J.shv[m]);
}

// ------------------------------------------------------------------------
// Face kernels, templated on the tile shape TW x TH (threads in x, y).
//
// x faces.  Tile (bx, by) of a job: Fortran cells c = (TW-1)*bx + tx
// (tx = 0..TW-1, c in 0..nx+1; c = 0 is the ghost of nx, c = nx+1 the ghost
// of 1), rows j = TH*by + 1 + ty.  Thread (tx, ty) reconstructs cell (c, j)
// and, for tx < TW-1, computes face f = c between cells c and c+1
// (f = 0..nx).  The positivity limiter runs for c = 0..nx only
// (src/finitevolume.f90:670), so face f = nx uses the unlimited left value
// of cell nx+1 while f = 0 uses the limited one of cell 1: the two values of
// the periodic seam.  Every face is computed by exactly one thread with the
// same arithmetic whatever the shape, so the results do not depend on it.
// ------------------------------------------------------------------------
template <int TW, int TH>
struct FaceTile {
  static constexpr int NT = TW * TH;               // threads
  static constexpr int VW = TW + 4, VH = TH + 4;   // halo tile of primitives
  static constexpr int NV = VW * VH;
  // first-sweep results per variable: VH x TW (x faces) or TH x VW (y faces)
  static constexpr int NQ = (TW * VH > TH * VW) ? TW * VH : TH * VW;
  // doubles of LDS: primitives + both first sweeps, reused for the WM exchange
  static constexpr int LDS = (3 * NV + 6 * NQ > 12 * NT) ? 3 * NV + 6 * NQ : 12 * NT;
};

// Gauss sum of the Rusanov fluxes of one face (src/finitevolume.f90:546-640)
// with the reference's operations one by one, between WP of the cell below the
// face and wm of the one above it (value a of 12 at wm[a * stride]).
template <bool X>
__device__ __forceinline__ void face_flux_general(const JobDev& J, const double WP[3][4],
                                                  const double* wm, int stride, double& acc1,
                                                  double& acc2, double& acc3) {
  acc1 = acc2 = acc3 = 0.0;
#pragma unroll 1
  for (int g = 0; g < 4; ++g) {
    double F1, F2, F3;
    // the Gauss point's values by selects: WP stays in registers
    double wp[3];
#pragma unroll
    for (int v = 0; v < 3; ++v)
      wp[v] = g == 0 ? WP[v][0] : g == 1 ? WP[v][1] : g == 2 ? WP[v][2] : WP[v][3];
    rusanov<X ? 1 : 0, X ? 0 : 1, X ? 0 : -1, X ? 1 : 0>(wp[0], wp[1], wp[2], wm[g * stride],
                                                         wm[(4 + g) * stride],
                                                         wm[(8 + g) * stride], J.g, F1, F2, F3);
    acc1 = acc1 + J.wbnd[g] * F1;
    acc2 = acc2 + J.wbnd[g] * F2;
    acc3 = acc3 + J.wbnd[g] * F3;
  }
}

// The same sum.  The regular form holds for finite states with
// depths in range (irregular = 0); a state that is not finite shows in one of
// its sums, and the face is then taken again with the reference's operations
// one by one.
template <bool X>
__device__ __forceinline__ void face_flux(const JobDev& J, const double WP[3][4],
                                          const double* wm, int stride, int irregular,
                                          double& acc1, double& acc2, double& acc3) {
  constexpr int N = X ? 1 : 2, T = X ? 2 : 1;  // normal and tangential velocity
  if (!irregular) {
    double a1 = 0.0, an = 0.0, at = 0.0;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      double F1, Fn, Ft;
      rusanov_regular(WP[0][g], WP[N][g], WP[T][g], wm[g * stride], wm[(4 * N + g) * stride],
                      wm[(4 * T + g) * stride], J.g, F1, Fn, Ft);
      a1 = a1 + J.wbnd[g] * F1;
      an = an + J.wbnd[g] * Fn;
      at = at + J.wbnd[g] * Ft;
    }
    acc1 = a1;
    acc2 = X ? an : at;
    acc3 = X ? at : an;
    if ((int)is_finite(a1) & (int)is_finite(an) & (int)is_finite(at)) return;
  }
  face_flux_general<X>(J, WP, wm, stride, acc1, acc2, acc3);
}

template <int TW, int TH>
__device__ __forceinline__ void x_faces(double* smem, int& irregular, const JobDev& J, int tile,
                                        int m, int slot, const NodeList& L) {
  using FT = FaceTile<TW, TH>;
  constexpr int NT = FT::NT, VW = FT::VW, VH = FT::VH, NV = FT::NV;
  constexpr int NQ = VH * TW;  // first sweeps per variable: VH rows x TW cells
  double* sV = smem;            // [3][VH rows][VW cols]
  double* sQM = smem + 3 * NV;  // [3][VH rows][TW cols]
  double* sQP = sQM + 3 * NQ;
  const int nx = J.nx, ny = J.ny;
  const int ntx = cdiv_d(nx + 1, TW - 1);
  const int tid = threadIdx.x, tx = tid % TW, ty = tid / TW;
  const int c0 = (tile % ntx) * (TW - 1);
  const int j0 = (tile / ntx) * TH + 1;
  const gdouble *h, *hu, *hv;
  node_state(J, m, h, hu, hv);
  // g h stays in the range of sqrt_regular for the depths of depths_regular
  if (tid == 0) irregular = !(J.g >= 0x1p-60 && J.g <= 0x1p60);

  for (int t = tid; t < NV; t += NT) {
    int lx = t % VW, ly = t / VW;
    size_t k = (size_t)wrap1(j0 - 2 + ly, ny) * nx + wrap1(c0 - 2 + lx, nx);
    double hh = h[k], u, v;
    cons_to_prim(hh, hu[k], hv[k], u, v);
    sV[t] = hh;
    sV[NV + t] = u;
    sV[2 * NV + t] = v;
  }
  __syncthreads();
  for (int t = tid; t < 3 * NQ; t += NT) {
    int var = t / NQ, r = t % NQ, ly = r / TW, lx = r % TW;
    const double* q = sV + var * NV + ly * VW + lx;
    double wm, wp;
    weno5_first(q[0], q[1], q[2], q[3], q[4], wm, wp);
    sQM[var * NQ + r] = wm;
    sQP[var * NQ + r] = wp;
  }
  __syncthreads();
  double WM[3][4], WP[3][4];
#pragma unroll
  for (int var = 0; var < 3; ++var) {
    const double* qm = sQM + var * NQ + ty * TW + tx;
    weno5_second(qm[0], qm[TW], qm[2 * TW], qm[3 * TW], qm[4 * TW], WM[var]);
    const double* qp = sQP + var * NQ + ty * TW + tx;
    weno5_second(qp[0], qp[TW], qp[2 * TW], qp[3 * TW], qp[4 * TW], WP[var]);
  }
  const int c = c0 + tx;
  if (J.recfix) {
    // ReconstructionFix 1 or 2 on the cells the shock indicator flags.
    // ShocksIndicatorX writes each cell's verdict to Ind(1, ii-1:ii+1, jj) in
    // loop order (src/shocksindicator.f90:50-55), so the last writer wins:
    // Ind(1, c, j) = Shock(min(c + 1, nx), j), from the depths at columns
    // min(c + 1, nx) - 1 .. + 1, all inside the halo tile.
    const int lc = min(c + 1, nx) - c0 + 2;
    const double* hrow = sV + (ty + 2) * VW;
    if (jameson_shock(hrow[lc - 1], hrow[lc], hrow[lc + 1])) {
#pragma unroll
      for (int var = 0; var < 3; ++var) {
        const double* q = sV + var * NV + (ty + 2) * VW + tx + 2;
        reconstruction_fix(J.recfix, q[-1], q[0], q[1], J.dx, WM[var], WP[var]);
      }
    }
  }
  const double vh = sV[(ty + 2) * VW + tx + 2];
  double mn = vh;
  if (c <= nx) {
    mn = positivity_limit(vh, J.wbnd, WM[0], WP[0]);
  } else {  // the unlimited ghost: only its WM is used
#pragma unroll
    for (int g = 0; g < 4; ++g) mn = min_n(mn, WM[0][g]);
  }
  if (!depths_regular(vh, mn)) irregular = 1;
  __syncthreads();
  double* sWM = smem;  // [12][NT]
#pragma unroll
  for (int a = 0; a < 12; ++a) sWM[a * NT + tid] = WM[a >> 2][a & 3];
  __syncthreads();
  const int j = j0 + ty;
  if (tx < TW - 1 && c <= nx && j <= ny) {
    double acc1, acc2, acc3;
    face_flux<true>(J, WP, sWM + tid + 1, NT, irregular, acc1, acc2, acc3);
    size_t o = (size_t)(j - 1) * (nx + 1) + c;
    if (J.wb && !L.wb_init) {  // FX = FX - FXWB (src/finitevolume.f90:485-486)
      acc1 = acc1 - G(J.FXWB[0])[o];
      acc2 = acc2 - G(J.FXWB[1])[o];
      acc3 = acc3 - G(J.FXWB[2])[o];
    }
    G(J.FX[slot][0])[o] = acc1;
    G(J.FX[slot][1])[o] = acc2;
    G(J.FX[slot][2])[o] = acc3;
  }
}

// ------------------------------------------------------------------------
// y faces: the transpose of x_faces.  Tile (bx, by): columns
// i = TW*bx + 1 + tx, Fortran rows r = (TH-1)*by + ty (0..ny+1); face g = r.
// ------------------------------------------------------------------------
template <int TW, int TH>
__device__ __forceinline__ void y_faces(double* smem, int& irregular, const JobDev& J, int tile,
                                        int m, int slot, const NodeList& L) {
  using FT = FaceTile<TW, TH>;
  constexpr int NT = FT::NT, VW = FT::VW, NV = FT::NV;
  constexpr int NQ = TH * VW;  // first sweeps per variable: TH rows x VW columns
  double* sV = smem;            // [3][VH rows][VW cols]
  double* sQM = smem + 3 * NV;  // [3][TH rows][VW cols]
  double* sQP = sQM + 3 * NQ;
  const int nx = J.nx, ny = J.ny;
  const int ntx = cdiv_d(nx, TW);
  const int tid = threadIdx.x, tx = tid % TW, ty = tid / TW;
  const int i0 = (tile % ntx) * TW + 1;
  const int r0 = (tile / ntx) * (TH - 1);
  const gdouble *h, *hu, *hv;
  node_state(J, m, h, hu, hv);
  // g h stays in the range of sqrt_regular for the depths of depths_regular
  if (tid == 0) irregular = !(J.g >= 0x1p-60 && J.g <= 0x1p60);

  for (int t = tid; t < NV; t += NT) {
    int lx = t % VW, ly = t / VW;
    size_t k = (size_t)wrap1(r0 - 2 + ly, ny) * nx + wrap1(i0 - 2 + lx, nx);
    double hh = h[k], u, v;
    cons_to_prim(hh, hu[k], hv[k], u, v);
    sV[t] = hh;
    sV[NV + t] = u;
    sV[2 * NV + t] = v;
  }
  __syncthreads();
  for (int t = tid; t < 3 * NQ; t += NT) {
    int var = t / NQ, r = t % NQ, ly = r / VW, lx = r % VW;
    const double* q = sV + var * NV + ly * VW + lx;
    double wm, wp;
    weno5_first(q[0], q[VW], q[2 * VW], q[3 * VW], q[4 * VW], wm, wp);
    sQM[var * NQ + r] = wm;
    sQP[var * NQ + r] = wp;
  }
  __syncthreads();
  double WM[3][4], WP[3][4];
#pragma unroll
  for (int var = 0; var < 3; ++var) {
    const double* qm = sQM + var * NQ + ty * VW + tx;
    weno5_second(qm[0], qm[1], qm[2], qm[3], qm[4], WM[var]);
    const double* qp = sQP + var * NQ + ty * VW + tx;
    weno5_second(qp[0], qp[1], qp[2], qp[3], qp[4], WP[var]);
  }
  const int r = r0 + ty;
  if (J.recfix) {
    // Ind(2, i, r) = Shock(i, min(r + 1, ny)) (src/shocksindicator.f90:84-89),
    // as in x_faces
    const int lr = min(r + 1, ny) - r0 + 2;
    const double* hcol = sV + tx + 2;
    if (jameson_shock(hcol[(lr - 1) * VW], hcol[lr * VW], hcol[(lr + 1) * VW])) {
#pragma unroll
      for (int var = 0; var < 3; ++var) {
        const double* q = sV + var * NV + (ty + 2) * VW + tx + 2;
        reconstruction_fix(J.recfix, q[-VW], q[0], q[VW], J.dy, WM[var], WP[var]);
      }
    }
  }
  const double vh = sV[(ty + 2) * VW + tx + 2];
  double mn = vh;
  if (r <= ny) {
    mn = positivity_limit(vh, J.wbnd, WM[0], WP[0]);
  } else {  // the unlimited ghost: only its WM is used
#pragma unroll
    for (int g = 0; g < 4; ++g) mn = min_n(mn, WM[0][g]);
  }
  if (!depths_regular(vh, mn)) irregular = 1;
  __syncthreads();
  double* sWM = smem;  // [12][NT]
#pragma unroll
  for (int a = 0; a < 12; ++a) sWM[a * NT + tid] = WM[a >> 2][a & 3];
  __syncthreads();
  const int i = i0 + tx;
  if (ty < TH - 1 && r <= ny && i <= nx) {
    double acc1, acc2, acc3;
    face_flux<false>(J, WP, sWM + tid + TW, NT, irregular, acc1, acc2, acc3);
    size_t o = (size_t)r * nx + (i - 1);
    if (J.wb && !L.wb_init) {  // FY = FY - FYWB (src/finitevolume.f90:487-488)
      acc1 = acc1 - G(J.FYWB[0])[o];
      acc2 = acc2 - G(J.FYWB[1])[o];
      acc3 = acc3 - G(J.FYWB[2])[o];
    }
    G(J.FY[slot][0])[o] = acc1;
    G(J.FY[slot][1])[o] = acc2;
    G(J.FY[slot][2])[o] = acc3;
  }
}

// ------------------------------------------------------------------------
// The faces of small grids, x (X) or y: two lanes per cell, one for the values
// at its lower face (WM) and one for those at its upper face (WP), on half
// tiles of 16 cells along the faces' normal (a) and 8 across (b).  Where a
// launch has fewer tiles than the device has CUs the time is that of one wave
// (a 16x16 tile: 1.3 us of loads, 1.9 of first sweeps, 4.7 of second sweeps,
// 1.8 of limiter and fluxes); here a lane has three second sweeps instead of
// six and two of the four Gauss points' fluxes, and idle CUs take the second
// half of the tile.  The lanes of a cell are neighbours, and so are the two
// lanes of a face (WP of cell a, WM of cell a + 1).
// ------------------------------------------------------------------------
constexpr int kSplitA = 16, kSplitB = 8;
constexpr int kDppPair = 0xB1;     // quad_perm [1,0,3,2]: the cell's other lane
constexpr int kDppNext = 0x130;    // wave_shl:1: the next lane

// positivity_limit with wm in even lanes (side 0) and wp in odd ones.
__device__ __forceinline__ double positivity_limit_pair(double vh, const double wbnd[4],
                                                        double w[4], int side) {
  double sum = wbnd[0] * w[0], mn = w[0];
#pragma unroll
  for (int g = 1; g < 4; ++g) {
    sum = sum + wbnd[g] * w[g];
    mn = min_n(mn, w[g]);
  }
  const double other = dpp<kDppPair, 0xf>(sum);
  const double alpha = side ? other : sum, beta = side ? sum : other;
  constexpr double c = 1. - 2. * kWLobatto;
  const double csi = div_pos(vh - kWLobatto * alpha - kWLobatto * beta, c, 1. / c);
  mn = min_n(min_n(mn, dpp<kDppPair, 0xf>(mn)), csi);
  const double num = vh - kMinDepth;
  double theta[4] = {1., 1., 1., 1.};
  // the same numbers, and so the same branch, in both lanes of the cell
  if (!((int)(fabs(num) >= fabs(vh - csi)) & (int)(fabs(num) >= fabs(vh - mn)))) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const double o = dpp<kDppPair, 0xf>(w[g]);
      const double mmin = min_r(min_r(csi, side ? o : w[g]), side ? w[g] : o);
      const double den = vh - mmin;
      if (vh == mmin)
        theta[g] = 1.;
      else if ((int)(fabs(num) >= fabs(den)) & (int)(fabs(num) <= kHuge))
        theta[g] = 1.;
      else
        theta[g] = min_r(1., fabs(num / den));
    }
  }
#pragma unroll
  for (int g = 0; g < 4; ++g) w[g] = vh + theta[g] * (w[g] - vh);
  return mn;
}

template <bool X>
__device__ __forceinline__ void split_faces(double* smem, int& irregular, const JobDev& J,
                                            int tile, int m, int slot, const NodeList& L) {
  constexpr int TA = kSplitA, TB = kSplitB, NT = 2 * TA * TB;
  constexpr int VA = TA + 4, VB = TB + 4, NV = VA * VB, NQ = VB * TA;
  double* sV = smem;            // [3][VB][VA]
  double* sQM = smem + 3 * NV;  // [3][VB][TA]
  double* sQP = sQM + 3 * NQ;
  const int nx = J.nx, ny = J.ny, na = X ? nx : ny, nb = X ? ny : nx;
  const int nta = cdiv_d(na + 1, TA - 1);
  const int tid = threadIdx.x, side = tid & 1, ca = (tid >> 1) % TA, cb = (tid >> 1) / TA;
  const int a0 = (tile % nta) * (TA - 1), b0 = (tile / nta) * TB + 1;
  const gdouble *h, *hu, *hv;
  node_state(J, m, h, hu, hv);
  if (tid == 0) irregular = !(J.g >= 0x1p-60 && J.g <= 0x1p60);

  if (tid < NV) {
    // x fastest
    const int va = X ? tid % VA : tid / VB, vb = X ? tid / VA : tid % VB;
    const int ia = wrap1(a0 - 2 + va, na), ib = wrap1(b0 - 2 + vb, nb);
    const size_t k = X ? (size_t)ib * nx + ia : (size_t)ia * nx + ib;
    double hh = h[k], u, v;
    cons_to_prim(hh, hu[k], hv[k], u, v);
    const int t = vb * VA + va;
    sV[t] = hh;
    sV[NV + t] = u;
    sV[2 * NV + t] = v;
  }
  static_assert(NV <= NT, "one cell of the halo tile per thread");
  __syncthreads();
  for (int t = tid; t < 3 * NQ; t += NT) {
    const int var = t / NQ, r = t % NQ;
    const double* q = sV + var * NV + (r / TA) * VA + r % TA;
    double wm, wp;
    weno5_first(q[0], q[1], q[2], q[3], q[4], wm, wp);
    sQM[t] = wm;
    sQP[t] = wp;
  }
  __syncthreads();
  double W[3][4];
#pragma unroll
  for (int var = 0; var < 3; ++var) {
    const double* q = (side ? sQP : sQM) + var * NQ + cb * TA + ca;
    weno5_second(q[0], q[TA], q[2 * TA], q[3 * TA], q[4 * TA], W[var]);
  }
  const int c = a0 + ca;
  const double* cell = sV + (cb + 2) * VA + ca + 2;
  if (J.recfix) {  // as in x_faces
    const double* hrow = sV + (cb + 2) * VA;
    const int lc = min(c + 1, na) - a0 + 2;
    if (jameson_shock(hrow[lc - 1], hrow[lc], hrow[lc + 1])) {
#pragma unroll
      for (int var = 0; var < 3; ++var) {
        const double* q = cell + var * NV;
        double fm[4], fp[4];
        reconstruction_fix(J.recfix, q[-1], q[0], q[1], X ? J.dx : J.dy, fm, fp);
#pragma unroll
        for (int g = 0; g < 4; ++g) W[var][g] = side ? fp[g] : fm[g];
      }
    }
  }
  const double vh = cell[0];
  double mn = vh;
  if (c <= na) {
    mn = positivity_limit_pair(vh, J.wbnd, W[0], side);
  } else {  // the unlimited ghost: only its WM is used
#pragma unroll
    for (int g = 0; g < 4; ++g) mn = min_n(mn, W[0][g]);
    if (side) mn = vh;
  }
  if (!depths_regular(vh, mn)) irregular = 1;
  __syncthreads();
  double* sW = smem;  // [12][NT]
#pragma unroll
  for (int a = 0; a < 12; ++a) sW[a * NT + tid] = W[a >> 2][a & 3];
  __syncthreads();
  // Gauss points 0, 1 of a face in its lower lane (WP), 2, 3 in its upper one
  constexpr int N = X ? 1 : 2, T = X ? 2 : 1;  // normal and tangential velocity
  const double* across = sW + (side ? min(tid + 1, NT - 1) : max(tid - 1, 0));
  double P1[2], Pn[2], Pt[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int g = side ? q : 2 + q;
    double own[3], far[3];
#pragma unroll
    for (int v = 0; v < 3; ++v) {
      own[v] = side ? W[v][q] : W[v][2 + q];
      far[v] = across[(4 * v + g) * NT];
    }
    double F1, Fn, Ft;
    rusanov_regular(side ? own[0] : far[0], side ? own[N] : far[N], side ? own[T] : far[T],
                    side ? far[0] : own[0], side ? far[N] : own[N], side ? far[T] : own[T], J.g,
                    F1, Fn, Ft);
    const double wg = side ? J.wbnd[q] : J.wbnd[2 + q];
    P1[q] = wg * F1;
    Pn[q] = wg * Fn;
    Pt[q] = wg * Ft;
  }
  double acc1 = 0.0, accn = 0.0, acct = 0.0;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    acc1 = acc1 + P1[q];
    accn = accn + Pn[q];
    acct = acct + Pt[q];
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {  // the upper lane's points
    acc1 = acc1 + dpp<kDppNext, 0xf>(P1[q]);
    accn = accn + dpp<kDppNext, 0xf>(Pn[q]);
    acct = acct + dpp<kDppNext, 0xf>(Pt[q]);
  }
  const int bb = b0 + cb;
  if (!side || ca >= TA - 1 || c > na || bb > nb) return;
  double acc2 = X ? accn : acct, acc3 = X ? acct : accn;
  if (irregular | !((int)is_finite(acc1) & (int)is_finite(acc2) & (int)is_finite(acc3)))
    face_flux_general<X>(J, W, sW + tid + 1, NT, acc1, acc2, acc3);
  const size_t o = X ? (size_t)(bb - 1) * (nx + 1) + c : (size_t)c * nx + (bb - 1);
  double* const* B = X ? J.FXWB : J.FYWB;
  double* const* F = X ? J.FX[slot] : J.FY[slot];
  if (J.wb && !L.wb_init) {  // less the well-balanced state's (src/finitevolume.f90:485-488)
    acc1 = acc1 - G(B[0])[o];
    acc2 = acc2 - G(B[1])[o];
    acc3 = acc3 - G(B[2])[o];
  }
  G(F[0])[o] = acc1;
  G(F[1])[o] = acc2;
  G(F[2])[o] = acc3;
}

// ------------------------------------------------------------------------
// Source term of a tile of TW x TH cells (1-based i = TW*bx + 1 + tx, j =
// TH*by + 1 + ty).  SourceTerms (src/equation.f90:352-388): h point values at
// the 4x4 Gauss points from a WENO5 second sweep along y (columns i-2..i+2)
// followed by one along x per y Gauss point; SW = -g*h*db; S = sum over x-GP
// (outer), y-GP (inner) of W*SW.
// ------------------------------------------------------------------------
template <int TW, int TH>
__device__ __forceinline__ void source_tile(double* smem, const JobDev& J, int tile, int m,
                                            double& S2, double& S3) {
  constexpr int NT = TW * TH, VW = TW + 4, VH = TH + 4, NV = VW * VH, NQ = VW * TH;
  double* sH = smem;        // [VH rows][VW cols]
  double* sVt = smem + NV;  // [yg][TH rows][VW cols]
  const int nx = J.nx, ny = J.ny;
  const int ntx = cdiv_d(nx, TW);
  const int tid = threadIdx.x, tx = tid % TW, ty = tid / TW;
  const int i0 = (tile % ntx) * TW + 1, j0 = (tile / ntx) * TH + 1;
  const int i = i0 + tx, j = j0 + ty;
  const size_t n = (size_t)J.n;
  const gdouble *h, *hu, *hv;
  node_state(J, m, h, hu, hv);
  for (int t = tid; t < NV; t += NT) {
    int lx = t % VW, ly = t / VW;
    sH[t] = h[(size_t)wrap1(j0 - 2 + ly, ny) * nx + wrap1(i0 - 2 + lx, nx)];
  }
  __syncthreads();
  for (int t = tid; t < NQ; t += NT) {
    const double* qh = sH + t;  // row ly, column lx of the halo tile
    double w[4];
    weno5_second(qh[0], qh[VW], qh[2 * VW], qh[3 * VW], qh[4 * VW], w);
#pragma unroll
    for (int yg = 0; yg < 4; ++yg) sVt[yg * NQ + t] = w[yg];
  }
  __syncthreads();
  if (i > nx || j > ny) return;
  const size_t k = (size_t)(j - 1) * nx + (i - 1);
  double hgp[4][4];  // [yg][xg]
#pragma unroll
  for (int yg = 0; yg < 4; ++yg) {
    const double* qv = sVt + yg * NQ + ty * VW + tx;
    weno5_second(qv[0], qv[1], qv[2], qv[3], qv[4], hgp[yg]);
  }
  S2 = 0.0;
  S3 = 0.0;
#pragma unroll
  for (int xg = 0; xg < 4; ++xg)
#pragma unroll
    for (int yg = 0; yg < 4; ++yg) {
      double hh = hgp[yg][xg];
      double bx = G(J.bx)[(size_t)(yg * 4 + xg) * n + k];
      double by = G(J.by)[(size_t)(yg * 4 + xg) * n + k];
      double sw2 = -J.g * hh * bx;
      double sw3 = -J.g * hh * by;
      S2 = S2 + J.wgp[xg][yg] * sw2;
      S3 = S3 + J.wgp[xg][yg] * sw3;
    }
}

// ------------------------------------------------------------------------
// The face fluxes of one FVTimeDerivative for up to three nodes and, in small
// launches, the sources: x-face, y-face and source tiles of every job in one
// launch, the three kinds being independent of each other.  On grids that do
// not fill the device they then run side by side (32^2: 11.8 us for 11.3 + 10.6
// one after the other, 7.9 with two lanes per cell; 128^2 lake: 22 us with the
// sources).  Launches that
// fill it several times over gain nothing from that, and their sources run
// better with the update (k_fvtd_source_update).
//
// Blocks come in groups of 8, one per XCD (workgroups are dealt round-robin to
// the 8 XCDs).  The sources' groups are spread evenly between the faces', and
// the L.count nodes of a source tile are 8 blocks apart: on one XCD and close
// together in time, so that the tile's bathymetry and well-balanced tables
// come from HBM once and from that XCD's L2 for the other nodes.
// ------------------------------------------------------------------------
struct FvtdTiles {
  const TileRef *xt, *yt, *st;
  int nxt, nyt, nst;
};

template <int XW, int XH, int YW, int YH, int SW, int SH, bool SPLIT = false>
__global__ __launch_bounds__(SW * SH, 4) void k_fvtd(EngineArgs E, FvtdTiles T, NodeList L) {
  static_assert(XW * XH * (SPLIT ? 2 : 1) == SW * SH && YW * YH * (SPLIT ? 2 : 1) == SW * SH,
                "one block size");
  constexpr int LX = SPLIT ? 12 * SW * SH : FaceTile<XW, XH>::LDS;
  constexpr int LY = SPLIT ? LX : FaceTile<YW, YH>::LDS;
  constexpr int LS = (SW + 4) * (SH + 4) + 4 * (SW + 4) * SH;
  __shared__ double smem[LX > LY ? (LX > LS ? LX : LS) : (LY > LS ? LY : LS)];
  __shared__ int irregular;  // a cell whose depths sqrt_regular may not take
  const int faces = (T.nxt + T.nyt) * L.count;
  const int gf = (faces + 7) / 8, gs = (T.nst + 7) / 8 * L.count;
  const int g = blockIdx.x / 8, r = blockIdx.x % 8;
  const int s0 = (int)((long long)g * gs / (gf + gs));  // source groups before this one
  const bool src = (int)((long long)(g + 1) * gs / (gf + gs)) > s0;
  if (src) {
    const int t = s0 / L.count * 8 + r, node = s0 % L.count;
    if (t >= T.nst) return;
    const TileRef R = tile_of(E, T.st, t);
    const JobDev& J = E.jobs[R.job];
    if (skipped_stage(E, R.job)) return;
    double S2, S3;
    source_tile<SW, SH>(smem, J, R.tile, L.m[node], S2, S3);
    const int ntx = cdiv_d(J.nx, SW);
    const int ci = (R.tile % ntx) * SW + threadIdx.x % SW;
    const int cj = (R.tile / ntx) * SH + threadIdx.x / SW;
    if (ci >= J.nx || cj >= J.ny) return;
    const int k = cj * J.nx + ci, out = L.out[node];
    if (J.wb && !L.wb_init) {
      S2 = S2 - G(J.SWB2)[k];
      S3 = S3 - G(J.SWB3)[k];
    }
    G(J.d2[out])[k] = S2;  // k_fvtd_update takes it from there
    G(J.d3[out])[k] = S3;
    return;
  }
  const int f = (g - s0) * 8 + r;
  if (f >= faces) return;
  const bool x = f < T.nxt * L.count;
  const int q = x ? f : f - T.nxt * L.count, nt = x ? T.nxt : T.nyt;
  const int node = q / nt;
  const TileRef R = tile_of(E, x ? T.xt : T.yt, q - node * nt);
  const JobDev& J = E.jobs[R.job];
  if (skipped_stage(E, R.job)) return;
  if constexpr (SPLIT) {
    static_assert(XW == kSplitA && XH == kSplitB && YH == kSplitA && YW == kSplitB, "the tiles");
    if (x)
      split_faces<true>(smem, irregular, J, R.tile, L.m[node], L.slot[node], L);
    else
      split_faces<false>(smem, irregular, J, R.tile, L.m[node], L.slot[node], L);
  } else if (x) {
    x_faces<XW, XH>(smem, irregular, J, R.tile, L.m[node], L.slot[node], L);
  } else {
    y_faces<YW, YH>(smem, irregular, J, R.tile, L.m[node], L.slot[node], L);
  }
}

// Divisions by a job's dx and dy through one reciprocal each.
struct OverDx {
  double dx, dy, rdx, rdy;
  bool shared;
  __device__ __forceinline__ explicit OverDx(const JobDev& J)
      : dx(J.dx), dy(J.dy), rdx(recip_refined(J.dx)), rdy(recip_refined(J.dy)),
        shared(recip_range(J.dx) & recip_range(J.dy)) {}
  __device__ __forceinline__ double x(double a) const {
    return shared ? div_pos(a, dx, rdx) : a / dx;
  }
  __device__ __forceinline__ double y(double a) const {
    return shared ? div_pos(a, dy, rdy) : a / dy;
  }
};

// Whether div_by may take every numerator seen: 0 or in [2^-400, 2^400]; the
// sign of a zero quotient is not kept.
struct Numerators {
  bool ok;
  __device__ __forceinline__ double operator()(double a) {
    const double m = fabs(a);
    ok = ok & (((int)(m >= kRecipLo) & (int)(m <= kRecipHi)) | (int)(a == 0.));
    return a;
  }
};

// ------------------------------------------------------------------------
// UpdateTimeDerivative (src/finitevolume.f90:446-540) of cell k = (ci, cj) from
// the fluxes in `slot` and its source S, into derivative slot o.
// ------------------------------------------------------------------------
__device__ __forceinline__ void update_cell(const JobDev& J, const NodeList& L, int o, int slot,
                                            int k, int ci, int cj, double S2, double S3) {
  const int nx = J.nx;
  if (L.wb_init) {  // building the well-balanced reference: keep S as SWB
    G(J.SWB2)[k] = S2;
    G(J.SWB3)[k] = S3;
    return;
  }
  const size_t fw = (size_t)cj * (nx + 1) + ci, fe = fw + 1;  // x faces
  const size_t gs = (size_t)cj * nx + ci, gn = gs + nx;       // y faces
  if (L.debug_S) {  // parity tests read S(2:3) from the first matrix scratch
    G(J.M[0][0])[k] = S2;
    G(J.M[0][1])[k] = S3;
  }
  // the face fluxes, with FXWB / FYWB already subtracted by the face kernels
  double fxe[3], fxw[3], fyn[3], fys[3];
#pragma unroll
  for (int v = 0; v < 3; ++v) {
    fxe[v] = G(J.FX[slot][v])[fe];
    fxw[v] = G(J.FX[slot][v])[fw];
    fyn[v] = G(J.FY[slot][v])[gn];
    fys[v] = G(J.FY[slot][v])[gs];
  }
  const OverDx over(J);
  // Ut(2:3) = S - (FX(i)-FX(i-1))/dx - (FY(j)-FY(j-1))/dy  (:525-527)
  const double ut2 = S2 - over.x(fxe[1] - fxw[1]) - over.y(fyn[1] - fys[1]);
  const double ut3 = S3 - over.x(fxe[2] - fxw[2]) - over.y(fyn[2] - fys[2]);
  if (L.ut1) {
    // the build without PATANKAR: Ut(1:3) (:529-533), with S(1) = 0 exactly
    // (SourceFunc's first component is 0., src/equation.f90:408)
    G(J.d1[o])[k] = 0.0 - over.x(fxe[0] - fxw[0]) - over.y(fyn[0] - fys[0]);
    G(J.d2[o])[k] = ut2;
    G(J.d3[o])[k] = ut3;
    return;
  }
  G(J.d2[o])[k] = ut2;  // FU2, FU3
  G(J.d3[o])[k] = ut3;
  // mass flux per face / dx: the production/destruction entries of
  // src/finitevolume.f90:496-523 are max(+-q, 0) and -min(+-q, 0) of these.
  G(J.qx[o])[fe] = over.x(fxe[0]);
  G(J.qy[o])[gn] = over.y(fyn[0]);
  if (ci == 0) G(J.qx[o])[fw] = over.x(fxw[0]);
  if (cj == 0) G(J.qy[o])[gs] = over.y(fys[0]);
}

// The update alone, one cell per thread, blockIdx.y = node; the sources of
// jobs with bathymetry are in the derivative slots already, less the
// well-balanced state's.  Bound by memory.
__global__ __launch_bounds__(256) void k_fvtd_update(EngineArgs E, const TileRef* blocks,
                                                     NodeList L) {
  const TileRef T = tile_of(E, blocks, blockIdx.x);
  const JobDev& J = E.jobs[T.job];
  if (skipped_stage(E, T.job)) return;
  const int o = L.out[blockIdx.y], nx = J.nx, k0 = T.tile * kCellBlock, k = k0 + threadIdx.x;
  if (k >= J.n) return;
  int ci, cj;
  cell_ij(k0 % nx, k0 / nx, threadIdx.x, nx, ci, cj);
  double S2 = 0.0, S3 = 0.0;
  if (J.bathy) {
    S2 = G(J.d2[o])[k];
    S3 = G(J.d3[o])[k];
  } else if (J.wb && !L.wb_init) {
    S2 = S2 - G(J.SWB2)[k];
    S3 = S3 - G(J.SWB3)[k];
  }
  update_cell(J, L, o, L.slot[blockIdx.y], k, ci, cj, S2, S3);
}

// Source and update in one pass over tiles of 16x16 cells, for launches large
// enough to fill the device without the sources beside the faces: the table
// loads of some blocks then overlap the WENO work of others at 5 waves per
// SIMD, and S needs no trip through memory (2048^2, 2.6 nodes on average: 700
// us, against 740 + 190 us for source tiles at the face kernels' 4 waves and
// the update alone).
__global__ __launch_bounds__(256) void k_fvtd_source_update(EngineArgs E, const TileRef* tiles,
                                                            int ntiles, NodeList L) {
  constexpr int TW = kTile, TH = kTile;
  __shared__ double smem[(TW + 4) * (TH + 4) + 4 * (TW + 4) * TH];
  const int grp = blockIdx.x / (8 * L.count), rem = blockIdx.x % (8 * L.count);
  const int node = rem / 8, t = grp * 8 + (rem % 8);
  if (t >= ntiles) return;
  const TileRef T = tile_of(E, tiles, t);
  const JobDev& J = E.jobs[T.job];
  if (skipped_stage(E, T.job)) return;
  const int ntx = cdiv_d(J.nx, TW);
  const int ci = (T.tile % ntx) * TW + threadIdx.x % TW;
  const int cj = (T.tile / ntx) * TH + threadIdx.x / TW;
  double S2 = 0.0, S3 = 0.0;
  if (J.bathy) source_tile<TW, TH>(smem, J, T.tile, L.m[node], S2, S3);
  if (ci >= J.nx || cj >= J.ny) return;
  const int k = cj * J.nx + ci;
  if (J.wb && !L.wb_init) {
    S2 = S2 - G(J.SWB2)[k];
    S3 = S3 - G(J.SWB3)[k];
  }
  update_cell(J, L, L.out[node], L.slot[node], k, ci, cj, S2, S3);
}

// ------------------------------------------------------------------------
// DeC momentum update, src/timediscretization.f90:531-543 (and :617-621,
// :717-721): Ua(m,2:3) = Ua(1,2:3); DO r=1,R: Ua(m) = Ua(m) + (dt*theta(m,r))*FUp(r)
// with R = MSteps.
// ------------------------------------------------------------------------
// One cell, the nodes m of systems s0..s1-1.  It runs inside the assembly kernel (the
// two read and write disjoint arrays), so that its loads overlap the
// assembly's latency-bound work.
template <int R>
__device__ __forceinline__ void momentum_cell(const JobDev& J, const SysList& S, int s0, int s1,
                                              int k, double dt, const double fu2[R],
                                              const double fu3[R]) {
  const double u0 = G(J.hu)[k], v0 = G(J.hv)[k];
  for (int s = s0; s < s1; ++s) {
    const int m = S.m[s];
    double u = u0, v = v0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const double c = dt * THETA[S.theta][m][r];
      u = u + c * fu2[r];
      v = v + c * fu3[r];
    }
    G(J.hun[m])[k] = u;
    G(J.hvn[m])[k] = v;
  }
}

// What the assembly and the momentum update of a cell take from the FVTDs: the
// mass fluxes / dx of its south, west, east and north faces at the R DeC nodes
// and Ut(2:3).  Node 0's are kept for all corrections, by the update or, FRESH =
// 2, by the first correction's assembly, for which all nodes are node 0 (`keep`;
// at_w, at_s: the cell has the first x or y face of its row or column).  With
// FRESH = 1 the other nodes' are formed here from the face fluxes and the source
// (as update_cell does), for a launch less per correction and, on large grids,
// a pass over memory (update + assembly without bathymetry: 900x800 98 -> 68 us,
// 1024^2 119 -> 99, 1500^2 331 -> 245, 2048^2 590 -> 448, three nodes; node 0:
// 32^2 11.3 -> 6.2, 257^2 17.6 -> 13.0, 1024^2 92 -> 78); all loads go out
// before the first quotient.
template <int R, int FRESH>
struct CellFluxes {
  double q[4][R], fu2[R], fu3[R];
  __device__ __forceinline__ CellFluxes(const JobDev& J, const SysList& S, int k, size_t fW,
                                        size_t gS, bool keep, bool at_w, bool at_s) {
    const size_t fE = fW + 1, gN = gS + J.nx;
    constexpr int R0 = FRESH == 2 ? 0 : 1;         // the nodes formed here
    constexpr int RL = FRESH == 2 ? 1 : R, R1 = FRESH ? RL : 1;
    double X[R1][2][2], Y[R1][2][2];  // [node][variable 2, 3][face]
#pragma unroll
    for (int r = 0; r < RL; ++r) {
      const bool here = FRESH && r >= R0;
      const gdouble* qx = G(here ? J.FX[r - R0][0] : J.qx[S.src[r]]);
      const gdouble* qy = G(here ? J.FY[r - R0][0] : J.qy[S.src[r]]);
      q[0][r] = qy[gS];
      q[1][r] = qx[fW];
      q[2][r] = qx[fE];
      q[3][r] = qy[gN];
      if (!here) {
        fu2[r] = G(J.FU2[S.src[r]])[k];
        fu3[r] = G(J.FU3[S.src[r]])[k];
      } else {
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          X[r % R1][v][0] = G(J.FX[r - R0][v + 1])[fW];
          X[r % R1][v][1] = G(J.FX[r - R0][v + 1])[fE];
          Y[r % R1][v][0] = G(J.FY[r - R0][v + 1])[gS];
          Y[r % R1][v][1] = G(J.FY[r - R0][v + 1])[gN];
        }
        fu2[r] = fu3[r] = 0.0;
        if (J.bathy) {  // node 0's sources are in slot 1: other blocks may still read
          fu2[r] = G(J.d2[FRESH == 2 ? kNode0Source : r])[k];  // them when FU2 is written
          fu3[r] = G(J.d3[FRESH == 2 ? kNode0Source : r])[k];
        } else if (J.wb) {
          fu2[r] = 0.0 - G(J.SWB2)[k];
          fu3[r] = 0.0 - G(J.SWB3)[k];
        }
      }
    }
    if (!FRESH) return;
    const OverDx over(J);
    Numerators seen{over.shared};
    double dX[R1][2], dY[R1][2];
#pragma unroll
    for (int r = R0; r < RL; ++r) {
      for (int f = 0; f < 4; ++f) seen(q[f][r]);
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        dX[r % R1][v] = seen(X[r % R1][v][1] - X[r % R1][v][0]);
        dY[r % R1][v] = seen(Y[r % R1][v][1] - Y[r % R1][v][0]);
      }
    }
    auto form = [&](auto ox, auto oy) {
#pragma unroll
      for (int r = R0; r < RL; ++r) {
        q[0][r] = oy(q[0][r]);
        q[1][r] = ox(q[1][r]);
        q[2][r] = ox(q[2][r]);
        q[3][r] = oy(q[3][r]);
        fu2[r] = fu2[r] - ox(dX[r % R1][0]) - oy(dY[r % R1][0]);
        fu3[r] = fu3[r] - ox(dX[r % R1][1]) - oy(dY[r % R1][1]);
      }
    };
    // The signs of zero quotients reach nothing: the sources are not -0, and
    // the mass fluxes are compared with 0 and taken by magnitude.
    if (__all(seen.ok))
      form([&](double a) { return div_by(a, over.dx, over.rdx); },
           [&](double a) { return div_by(a, over.dy, over.rdy); });
    else
      form([&](double a) { return over.x(a); }, [&](double a) { return over.y(a); });
    if (FRESH != 2) return;
    if (keep) {
      G(J.FU2[0])[k] = fu2[0];
      G(J.FU3[0])[k] = fu3[0];
      G(J.qx[0])[fE] = q[2][0];
      G(J.qy[0])[gN] = q[3][0];
      if (at_w) G(J.qx[0])[fW] = q[1][0];
      if (at_s) G(J.qy[0])[gS] = q[0][0];
    }
#pragma unroll
    for (int r = 1; r < R; ++r) {
#pragma unroll
      for (int f = 0; f < 4; ++f) q[f][r] = q[f][0];
      fu2[r] = fu2[0];
      fu3[r] = fu3[0];
    }
  }
};

// ------------------------------------------------------------------------
// Reductions
// ------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Deterministic sum over a 256-thread block, returned to every thread.
// red: 4 doubles of shared memory.
__device__ __forceinline__ double block_sum_all(double v, double* red) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[w] = v;
  __syncthreads();
  double r = ((red[0] + red[1]) + red[2]) + red[3];
  __syncthreads();
  return r;
}

// Sum of part[0..nb) in a fixed order by one 256-thread block, with 8
// independent loads in flight per thread.
__device__ double block_sum_array(const double* part, int nb, double* red) {
  double a[8] = {0., 0., 0., 0., 0., 0., 0., 0.};
  int b = threadIdx.x;
  for (; b + 7 * 256 < nb; b += 8 * 256) {
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] += part[b + u * 256];
  }
  for (int u = 0; b < nb; b += 256, ++u) a[u & 7] += part[b];
  double t = ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
  return block_sum_all(t, red);
}

// Decide `tol < SUM(d)/n` (src/jacobi_iteration.f90:71,77) where the
// reference sums the d_i >= 0 sequentially in row order and S is the same sum
// taken in parallel.  Both roundings differ from the exact sum by at most
// (n-1)u*sum(d), so whenever tol lies outside [S - B, S + B]/n with
// B = 8nuS the decision is that of the sequential sum; inside the window the
// caller recomputes the sequential sum exactly.  1 continue, 0 stop, -1 open.
__device__ __forceinline__ int certified_continue(double S, int n, double tol) {
  if (isnan(S)) return 0;
  if (isinf(S)) return 1;
  const double u = 1.1102230246251565e-16;  // 2^-53
  double B = 8.0 * (double)n * u * S;
  double lo = (S - B) / (double)n, hi = (S + B) / (double)n;
  if (tol < lo) return 1;
  if (!(tol < hi)) return 0;
  return -1;
}

// Exact replay of the reference's sequential residual: mode 0 sums
// |0 - a_i|, mode 1 sums |a_i - b_i|; divided by n.
__device__ double sequential_residual(int n, const double* a, const double* b, int mode) {
  double r = 0.0;
  for (int i = 0; i < n; ++i) r = r + (mode == 0 ? fabs(0.0 - a[i]) : fabs(a[i] - b[i]));
  return r / (double)n;
}

// ------------------------------------------------------------------------
// Patankar assembly (MODIFIED_PATANKAR_MATRIX_INVERSION,
// src/timediscretization.f90:795-887) fused with the first Jacobi sweep from
// x^0 = rhs (src/jacobi_iteration.f90:67-76).
// ------------------------------------------------------------------------
// PATANKAR_DIV of a zero numerator, without the division: the reference's
// 2*h*z/(h*h + MAX(h*h, 1e-6)) for z = +0 or -0 is +0 when h < MIN_DEPTH, z
// itself when h is finite (the quotient keeps the sign of z), and NaN when h
// is +Inf or NaN (2*h*z is then NaN) -- exactly what this returns.
__device__ __forceinline__ double patankar_div_zero(double z, double h) {
  return (h < kMinDepth) ? 0. : z * (h * 0. + 1.);
}

// The parts of PATANKAR_DIV (src/timediscretization.f90:913-924) that depend
// on the depth h alone: 2*h*prod/(h*h + MAX(h*h, MIN_DEPTH)) is (2h)*prod / den
// evaluated left to right, 0 when h < MIN_DEPTH; and its value for a +0 and a
// -0 numerator.
struct PdDepth {
  double twoh, den, zp, zm;
  bool dry;
};
__device__ __forceinline__ PdDepth pd_depth(double h) {
  PdDepth d;
  d.dry = h < kMinDepth;
  d.twoh = 2. * h;
  d.den = h * h + max_r(h * h, kMinDepth);
  d.zp = patankar_div_zero(0., h);
  d.zm = patankar_div_zero(-0., h);
  return d;
}

// PATANKAR_DIV(a, h) with h the neighbour's depth (useL) or the row's own.
// WET: no depth of the row is below MIN_DEPTH, so no quotient becomes 0.
template <bool WET>
__device__ __forceinline__ double pd_quot(bool useL, double a, const PdDepth& L,
                                          const PdDepth& K) {
  const double q = ((useL ? L.twoh : K.twoh) * a) / (useL ? L.den : K.den);
  return (!WET && (useL ? L.dry : K.dry)) ? 0. : q;
}

// One stencil slot of a row at the R DeC nodes (src/timediscretization.f90:
// 800-884): with P and De the slot's production and destruction,
//   theta > 0: M = M - c*PD(P, hL), D = D + c*PD(De, hK);
//   otherwise: D = D - c*PD(P, hK), M = M + c*PD(De, hL).
// s is the slot's oriented face mass flux: q = F/dx for the west and south
// slots, -q for the east and north ones, so that P = s > 0 ? s : +0 and
// De = s < 0 ? -s : -0 (src/finitevolume.f90:496-523).  At most one of P and
// De is nonzero, and the nonzero one is |s|, so each node needs one division;
// the zero one takes PdDepth's zp or zm, the value PATANKAR_DIV gives it.
// The sign of theta (bit r of pos) is the same for the whole launch, so the
// branch on it is uniform.
template <int R, bool WET>
__device__ __forceinline__ void patankar_slot(int pos, const double c[R], const double s[R],
                                              const PdDepth& L, const PdDepth& K, double& M,
                                              double& D) {
  M = 0.;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const double sr = s[r];
    const bool gt = sr > 0., lt = sr < 0.;
    if ((pos >> r) & 1) {  // L takes P, K takes De
      const double dv = pd_quot<WET>(gt, fabs(sr), L, K);
      const double tL = c[r] * (gt ? dv : L.zp);
      const double tK = c[r] * (lt ? dv : K.zm);
      M = M - tL;
      D = D + tK;
    } else {  // L takes De, K takes P
      const double dv = pd_quot<WET>(lt, fabs(sr), L, K);
      const double tL = c[r] * (lt ? dv : L.zm);
      const double tK = c[r] * (gt ? dv : K.zp);
      M = M + tL;
      D = D - tK;
    }
  }
}

// The four stencil slots of one row-system (sparse_matmul in CSR order S, W,
// self (value 0), E, N): hands the slots' matrix entries to put, accumulates the
// diagonal into D and returns the product with the neighbours' rhs values.
// sq: the row's column of the staged fluxes, NT apart.
template <int R, bool WET, int NT, class Put>
__device__ __forceinline__ double patankar_row(Put put, const double* sq, int pos,
                                               const double c[R], const PdDepth& pK, double hS,
                                               double hW, double hE, double hN, double bS,
                                               double bW, double bE, double bN, double b,
                                               double& D) {
  double p = 0.;
#pragma unroll 1
  for (int sl = 0; sl < 4; ++sl) {
    // the slot's neighbour values, selected from the ones loaded by the caller
    const double hL = sl == 0 ? hS : sl == 1 ? hW : sl == 2 ? hE : hN;
    const double bL = sl == 0 ? bS : sl == 1 ? bW : sl == 2 ? bE : bN;
    double q[R];
#pragma unroll
    for (int r = 0; r < R; ++r) q[r] = sq[(sl * R + r) * NT];
    double M;
    patankar_slot<R, WET>(pos, c, q, pd_depth(hL), pK, M, D);
    put(sl, M);
    p = p + M * bL;
    if (sl == 1) p = p + 0. * b;
  }
  return p;
}

// The denominators and right-hand side of the systems: hp(m,.) is h^n in the
// first correction and node m's depth after it; the rhs is h^n.  With
// S.hp_view both come from the buffers k_hp_view fills.
__device__ __forceinline__ const gdouble* system_hp(const JobDev& J, const SysList& S, int m) {
  return G(S.hp_view ? J.hres[3] : (S.hp_is_un ? J.h : J.hres[m]));
}
__device__ __forceinline__ const gdouble* system_rhs(const JobDev& J, const SysList& S) {
  return G(S.hp_view ? J.hres[2] : J.h);
}

// Block b's place among n (k_assemble's), for every XCD to work on one run of
// them (blocks are dealt round-robin to the 8 XCDs, each with an L2 of its
// own): the fluxes and depths of a cell's row neighbours are then read by the
// same XCD, a few blocks earlier or later (257^2 17.9 -> 15.7 us, 1024^2 80 ->
// 75.5, 2048^2 363 -> 351; k_sweep, with one stencil value per system, gained
// nothing).  Launched with xcd_blocks(n) blocks, those with places >= n to
// spare; few blocks are taken as they come.
constexpr int kXcdFrom = 64;
__device__ __forceinline__ int xcd_chunk(int b, int n) {
  return n < kXcdFrom ? b : (b & 7) * ((n + 7) / 8) + (b >> 3);
}
inline int xcd_blocks(int n) { return n < kXcdFrom ? n : (n + 7) / 8 * 8; }

// Cell blocks per block of the assembly with the first sweep, on large grids:
// the block's look-ups and its four sums over the block are shared by 1024
// cells, and k_decide, which reads all partial sums with one block at 14 bytes
// a nanosecond, has a quarter of them (2048^2: 410 + 34 -> 358 + 13 us; 1500^2:
// 226 + 23 -> 203 + 11).  k_sweep stays at a block per 256 cells: it is bound
// by its loads and lost as much (78 -> 93 us) as its decision gained.  Below
// 4096 cell blocks the device would be left idle, and the tables of several
// jobs name cell blocks one by one.
constexpr int kSumBlocks = 4, kSumBlocksFrom = 4096;
__host__ __device__ inline int sum_blocks(const EngineArgs& E, int nblk) {
  return E.single >= 0 && nblk >= kSumBlocksFrom ? kSumBlocks : 1;
}

// FIRST: the first sweep and its residual sums, for a launch per sweep; without
// it only the matrix, for k_solve.  blockIdx.y picks the system where the grid
// has that dimension (launch_assemble_matrix), else the block does them all.
template <int R, bool FIRST, int FRESH = 0>
__global__ __launch_bounds__(256) void k_assemble(EngineArgs E, const TileRef* blocks, int nblocks,
                                                  SysList S) {
  __shared__ double red[4];
  __shared__ double sq[4 * R * 256];  // [slot*R + node][thread]: face mass fluxes
  const int place = xcd_chunk(blockIdx.x, nblocks);
  if (place >= nblocks) return;
  const TileRef T = tile_of(E, blocks, place);
  const JobDev& J = E.jobs[T.job];
  if (skipped_stage(E, T.job)) return;
  const int nx = J.nx, ny = J.ny, n = J.n;
  const int tid = threadIdx.x;
  const double dt = E.status[T.job].dt;
  const int s0 = gridDim.y > 1 ? blockIdx.y : 0, s1 = gridDim.y > 1 ? s0 + 1 : S.count;
  const int per = FIRST ? sum_blocks(E, J.nblk) : 1;
  double dsum[kMaxSys] = {}, bsum = 0.;
#pragma unroll 1
  for (int g = 0; g < per; ++g) {
    const int tile = T.tile * per + g, k = tile * kCellBlock + tid;
    const bool in = k < n;
    int kS = 0, kW = 0, kE = 0, kN = 0;  // neighbours
    double b = 0., bS = 0., bW = 0., bE = 0., bN = 0.;
    if (in) {
      const int k0 = tile * kCellBlock;
      int i, j;
      cell_ij(k0 % nx, k0 / nx, tid, nx, i, j);
      kS = (j == 0 ? ny - 1 : j - 1) * nx + i;
      kW = j * nx + (i == 0 ? nx - 1 : i - 1);
      kE = j * nx + (i == nx - 1 ? 0 : i + 1);
      kN = (j == ny - 1 ? 0 : j + 1) * nx + i;
      const CellFluxes<R, FRESH> F(J, S, k, (size_t)j * (nx + 1) + i, (size_t)j * nx + i,
                                     s0 == 0, i == 0, j == 0);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        sq[(0 * R + r) * 256 + tid] = F.q[0][r];
        sq[(1 * R + r) * 256 + tid] = F.q[1][r];
        sq[(2 * R + r) * 256 + tid] = -F.q[2][r];  // east and north slots: the flux
        sq[(3 * R + r) * 256 + tid] = -F.q[3][r];  // oriented into the cell
      }
      const gdouble* rhs = system_rhs(J, S);
      if (FIRST) {
        b = rhs[k];
        bS = rhs[kS];
        bW = rhs[kW];
        bE = rhs[kE];
        bN = rhs[kN];
      }
      momentum_cell<R>(J, S, s0, s1, k, dt, F.fu2, F.fu3);
    }
    // One system at a time, and within it one stencil slot at a time (S, W, E,
    // N: the CSR order), so that only one slot's divisions are live.  Each
    // thread reads back only its own column of sq, so no barrier is needed.
#pragma unroll 1
    for (int s = s0; s < s1; ++s) {
      double d = 0.;
      if (in) {
        const int m = S.m[s];
        const gdouble* hp = system_hp(J, S, m);
        const double hK = hp[k], hS = hp[kS], hW = hp[kW], hE = hp[kE], hN = hp[kN];
        const PdDepth pK = pd_depth(hK);
        const int pos = THETA_POS[S.theta][m];
        double c[R];
#pragma unroll
        for (int r = 0; r < R; ++r) c[r] = dt * THETA[S.theta][m][r];
        // sol = (rhs - prod)/diag; rows of a wave with no depth below
        // MIN_DEPTH take the branch without the dry-depth selects
        double D = 1.;
        const bool dry = pK.dry | (hS < kMinDepth) | (hW < kMinDepth) | (hE < kMinDepth) |
                         (hN < kMinDepth);
        auto put = [&](int sl, double v) { G(J.M[s][sl])[k] = v; };
        const double p = __any(dry)
                             ? patankar_row<R, false, 256>(put, sq + tid, pos, c, pK, hS, hW, hE, hN,
                                                           bS, bW, bE, bN, b, D)
                             : patankar_row<R, true, 256>(put, sq + tid, pos, c, pK, hS, hW, hE, hN,
                                                          bS, bW, bE, bN, b, D);
        G(J.M[s][4])[k] = D;
        if (FIRST) {
          double x1 = (b - p) / D;
          G(J.xj[m][1])[k] = x1;
          d = fabs(x1 - b);
        }
      }
      if (!FIRST) continue;
#pragma unroll
      for (int q = 0; q < kMaxSys; ++q) dsum[q] += q == s ? d : 0.;
    }
    if (FIRST && in) bsum += fabs(0.0 - b);
  }
  if (!FIRST) return;
  const size_t nsum = cdiv_d(J.nblk, per);
#pragma unroll
  for (int s = 0; s < kMaxSys; ++s)
    if (s < S.count) {
      const double t = block_sum_all(dsum[s], red);
      if (tid == 0) J.part[s * nsum + T.tile] = t;
    }
  const double t = block_sum_all(bsum, red);
  if (tid == 0) J.part[kMaxSys * nsum + T.tile] = t;
}

// One Jacobi sweep of every still-active system (src/jacobi_iteration.f90:72-80).
__global__ __launch_bounds__(256) void k_sweep(EngineArgs E, const TileRef* blocks, SysList S) {
  __shared__ double red[4];
  const TileRef T = tile_of(E, blocks, blockIdx.x);
  const JobDev& J = E.jobs[T.job];
  if (skipped(E, T.job)) return;
  int act[kMaxSys] = {0, 0, 0}, cur[kMaxSys] = {0, 0, 0};
  bool any = false;
  for (int s = 0; s < S.count; ++s) {
    act[s] = E.status[T.job].st[s].active;
    cur[s] = E.status[T.job].st[s].cur;
    any = any || act[s];
  }
  if (!any) return;  // every system of this job has stopped
  const int nx = J.nx, ny = J.ny, n = J.n;
  const int k = T.tile * kCellBlock + threadIdx.x;
  double d[kMaxSys] = {0., 0., 0.};
  if (k < n) {
    const int k0 = T.tile * kCellBlock;
    int i, j;
    cell_ij(k0 % nx, k0 / nx, threadIdx.x, nx, i, j);
    const int kS = (j == 0 ? ny - 1 : j - 1) * nx + i;
    const int kN = (j == ny - 1 ? 0 : j + 1) * nx + i;
    const int kW = j * nx + (i == 0 ? nx - 1 : i - 1);
    const int kE = j * nx + (i == nx - 1 ? 0 : i + 1);
    const double b = system_rhs(J, S)[k];
    for (int s = 0; s < S.count; ++s) {
      if (!act[s]) continue;
      const int m = S.m[s];
      const gdouble* xo = G(J.xj[m][cur[s]]);
      gdouble* xn = G(J.xj[m][1 - cur[s]]);
      double p = 0.;
      p = p + G(J.M[s][0])[k] * xo[kS];
      p = p + G(J.M[s][1])[k] * xo[kW];
      p = p + 0. * xo[k];
      p = p + G(J.M[s][2])[k] * xo[kE];
      p = p + G(J.M[s][3])[k] * xo[kN];
      double xv = (b - p) / G(J.M[s][4])[k];
      xn[k] = xv;
      d[s] = fabs(xv - xo[k]);
    }
  }
  for (int s = 0; s < S.count; ++s) {
    if (!act[s]) continue;
    double t = block_sum_all(d[s], red);
    if (threadIdx.x == 0) J.part[(size_t)s * J.nblk + T.tile] = t;
  }
}

// Stop decision, one block per job: after the assembly (FIRST) or a sweep.
template <bool FIRST>
__global__ __launch_bounds__(256) void k_decide(EngineArgs E, const int* jobs, SysList S) {
  __shared__ double red[4];
  const int job = job_of(E, jobs, blockIdx.x);
  const JobDev& J = E.jobs[job];
  JobStatus* st = E.status + job;
  if (skipped(E, job)) return;
  const int n = J.n, nb = FIRST ? cdiv_d(J.nblk, sum_blocks(E, J.nblk)) : J.nblk;
  double tot[kMaxSys + 1] = {0., 0., 0., 0.};
  int act[kMaxSys] = {0, 0, 0}, cur[kMaxSys] = {0, 0, 0};
  for (int s = 0; s < S.count; ++s) {
    act[s] = FIRST ? 1 : st->st[s].active;
    cur[s] = FIRST ? 0 : st->st[s].cur;
  }
  for (int s = 0; s < S.count; ++s)
    if (act[s]) tot[s] = block_sum_array(J.part + (size_t)s * nb, nb, red);
  if (FIRST) tot[kMaxSys] = block_sum_array(J.part + (size_t)kMaxSys * nb, nb, red);
  if (threadIdx.x != 0) return;
  const double* rhs = S.hp_view ? J.hres[2] : J.h;
  if (FIRST) {
    // initial residual SUM(ABS(0 - rhs))/n, common to all systems
    int c0 = certified_continue(tot[kMaxSys], n, E.tol);
    int amb0 = 0;
    if (c0 < 0) {
      double r = sequential_residual(n, rhs, nullptr, 0);
      c0 = (E.tol < r) ? 1 : 0;
      amb0 = 1;
    }
    for (int s = 0; s < S.count; ++s) {
      JacState& q = st->st[s];
      q.ambiguous = amb0;
      q.cur = 1;
      if (!c0 || E.max_iter <= 0) {
        q.k = 0;
        q.active = 0;
        q.zero = 1;
        // no sweep: "not converged" when the initial residual is above the
        // tolerance (src/jacobi_iteration.f90:82-84)
        q.nonconv = c0 ? 1 : 0;
        q.residual = tot[kMaxSys] / (double)n;
        continue;
      }
      q.k = 1;
      q.zero = 0;
      int c1 = certified_continue(tot[s], n, E.tol);
      if (c1 < 0) {
        double r = sequential_residual(n, J.xj[S.m[s]][1], rhs, 1);
        c1 = (E.tol < r) ? 1 : 0;
        q.ambiguous += 1;
      }
      q.residual = tot[s] / (double)n;
      q.active = (c1 && q.k < E.max_iter) ? 1 : 0;
      q.nonconv = (c1 && !q.active) ? 1 : 0;
    }
  } else {
    for (int s = 0; s < S.count; ++s) {
      if (!act[s]) continue;
      JacState& q = st->st[s];
      q.k += 1;
      q.cur = 1 - cur[s];
      int c = certified_continue(tot[s], n, E.tol);
      if (c < 0) {
        const int m = S.m[s];
        double r = sequential_residual(n, J.xj[m][q.cur], J.xj[m][cur[s]], 1);
        c = (E.tol < r) ? 1 : 0;
        q.ambiguous += 1;
      }
      q.residual = tot[s] / (double)n;
      q.active = (c && q.k < E.max_iter) ? 1 : 0;
      q.nonconv = (c && !q.active) ? 1 : 0;
    }
  }
}

// ------------------------------------------------------------------------
// The Jacobi iteration of a correction's solves in one launch, for grids whose
// systems fit the register files.
//
// A block of 512 threads owns a tile of a system and holds it with a halo of
// kSolveWindow = 4 cells: a lane per column (64 with the halo) and a strip of
// up to 11 rows per wave, matrix rows and iterate in registers.  It sweeps 4
// times without looking at the other blocks -- each sweep spoils one more ring
// of the halo -- then the blocks exchange their outer 4 rings and the residual
// sums of the 4 sweeps, and the stop rule is applied to the sums in order.  A
// solve that stopped inside the window sweeps again from the window's start to
// that iterate.  The first window needs no exchange before it: it starts from
// the right-hand side, known everywhere.  So no sweep reads the matrix from
// memory, and no launch, host prediction or empty sweep is paid per sweep.
//
// Within a sweep a row's neighbours in the strip are the thread's own, those
// to the west and east come by DPP moves; LDS carries only the strips' first
// and last rows.  With the iterate in LDS a row took 5 reads and a write, and
// with the full division (solve_row) 45 instructions in place of 19: 2.1 ->
// 1.0 us a sweep of 11 rows per thread.  Small grids need one block (ALONE)
// with any number of columns and keep the iterate in LDS.
//
// Measured per launch, three systems unless said: 257^2 31.4 -> 23.9 us,
// 512^2 68 -> 53 us, one system of 1024^2 81 -> 64 us, 32^2 14.4 -> 13.5 us
// (iterate in LDS and full division before); a launch per sweep and one per
// stop decision took 190 us a correction at 32^2, 135 us at 257^2.  Of the
// 64 us at 1024^2 (10 sweeps) 14 are the loads of the matrix (69 MB, 5 TB/s),
// 15 the sweeps, 25 the three exchanges with their sums and halo loads.
// Windows of 6 with halos of 6 lose as much in the tiles as they save in
// exchanges (257^2: 27 us, 512^2: 60 us).
//
// The exchange goes through agent-scope atomic stores and loads, which bypass
// the XCDs' separate L2s, so no cache is written back: a block drains its
// stores (s_waitcnt vmcnt(0)), then publishes its sums in slots whose low 8
// bits carry the round's tag, and polls the other blocks' slots for that tag.
// Measured per round: 2.4 us for 8 blocks, 3.3 us for 64, 4.3 us for 240; with
// a counter instead of tags 3.0, 3.7, 6.7 us; with agent-scope fences 5.1 us
// for 64.  The cells of round t go to buffer t & 1: a block overwrites it in
// round t + 2, after every block has published round t + 1 and so finished
// reading round t.
//
// The tag takes the sum's low 8 bits, a relative change below 2^-44, which the
// stop rule allows for.  Tags count on over the launches
// (JobStatus::rounds), and a slot is rewritten in every second round of its
// form, so the tag it held before is the expected one less 2.
//
// The host launches no more blocks at once than the device holds
// concurrently, and no two such launches side by side.  A wait is bounded all
// the same: when it runs out (another process on the device, say), or a stop
// decision lies inside the certified window, the solve ends as kSolveOpen, the
// step is not committed and the host runs it again with the launches of one
// sweep each.  After a wait that ran out the tags of the blocks no longer agree:
// the job's solves that are on the stream already give up their first exchange
// at once (JobStatus::polls; looked at before the sweeps it cost 1 us a launch),
// and the host clears slots and rounds before the next one (engine_batch).
// ------------------------------------------------------------------------
__device__ __forceinline__ double agent_load(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void agent_store(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Sum over the wave in a fixed order, in every lane; six dependent steps
// without LDS (the shuffles of wave_sum are LDS instructions of 130 cycles).
__device__ __forceinline__ double wave_sum_dpp(double v) {
  v += dpp<0x111, 0xf>(v);  // row_shr:1
  v += dpp<0x112, 0xf>(v);
  v += dpp<0x114, 0xf>(v);
  v += dpp<0x118, 0xf>(v);
  v += dpp<0x142, 0xa>(v);  // row_bcast:15
  v += dpp<0x143, 0xc>(v);  // row_bcast:31
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                          __builtin_amdgcn_readlane(__double2loint(v), 63));
}

constexpr int kSolveRows = kSolveRpt[kSolveForms - 1] * kSolveThreads;  // of the largest tile
constexpr int kSolveWaves = kSolveThreads / 64;
constexpr int kSolveAloneRows = 4 * kSolveThreads;  // most rows of a block without others
static_assert(kSolveWaves == 8 && kSolveKinds <= 8, "the stop rule's lanes");

struct SolveShared {
  union {
    double x[3][kSolveAloneRows];  // ALONE: the iterate: the window's start and two buffers
    struct {
      double start[kSolveRows];            // the window's start, each thread's own rows
      double edge[2][kSolveWaves][2][64];  // the strips' first and last rows, by parity
    } t;
  };
  double red[kSolveKinds][kSolveWaves];
  double tot[kSolveKinds][4];
  int lost;
  // the round after which an iterate left the short form's range; ~0: a row is
  // outside it from the start
  unsigned irregular;
};

// Ranges in which a sweep needs none of the care for signed zeros, infinities
// and rescaled divisions: with off-diagonal entries in [-2^40, 0], a diagonal
// in [2^-8, 2^100], a right-hand side in [2^-200, 2^100] and an iterate in
// [0, 2^200] at the start of the window, every product is <= 0, every numerator
// in [2^-200, 2^392] and every quotient in [2^-300, 2^400] (a sweep lets the
// iterate grow by less than 2^50).  There 0. + p, + 0.*x change nothing, and
// the quotient has div_by's bits.
__device__ __forceinline__ bool solve_row_regular(const double M[4], double D, double b) {
  int ok = (int)(D >= 0x1p-8) & (int)(D <= 0x1p100) & (int)(b >= 0x1p-200) & (int)(b <= 0x1p100);
#pragma unroll
  for (int q = 0; q < 4; ++q) ok &= (int)(M[q] >= -0x1p40) & (int)(M[q] <= 0.);
  return ok;
}

// p, the same in every lane of the wave, in scalar registers.
template <class T>
__device__ __forceinline__ T* uniform(T* p) {
  const unsigned long long v = (unsigned long long)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
  return (T*)((unsigned long long)hi << 32 | lo);
}

constexpr unsigned kSolveStartHi = (1023u + 200u) << 20;  // high word of 2^200; signs lie above

// x_new of a row (src/jacobi_iteration.f90:72-80); R: recip_refined(D).
template <bool SHORT>
__device__ __forceinline__ double solve_row(const double M[4], double D, double R, double b,
                                            double x, double yS, double yW, double yE,
                                            double yN) {
  if (SHORT) {
    double p = M[0] * yS;
    p = p + M[1] * yW;
    p = p + M[2] * yE;
    p = p + M[3] * yN;
    return div_by(b - p, D, R);
  }
  double p = 0.;
  p = p + M[0] * yS;
  p = p + M[1] * yW;
  p = p + 0. * x;
  p = p + M[2] * yE;
  p = p + M[3] * yN;
  return (b - p) / D;
}

// ALONE: the whole grid in the block, no halo and no exchange.
template <int RPT, bool ALONE>
__device__ __forceinline__ void solve_block(SolveShared& L, const EngineArgs& E, const SolveRef W,
                                            const SysList& S, int limit, int first_solve) {
  constexpr int NT = kSolveThreads, HALO = ALONE ? 0 : kSolveWindow;
  const JobDev& J = E.jobs[W.job];
  const int tid = threadIdx.x, lane = tid & 63, s = W.sys, m = S.m[s];
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nx = J.nx, ny = J.ny, n = J.n;
  JobStatus* st = E.status + W.job;
  // own cells [ox, ox + ow) x [oy, oy + oh)
  int nb = 1, ox = 0, oy = 0, ow = nx, oh = ny;
  unsigned round0 = 0;
  int most = 0;  // polls
  if (!ALONE) {
    const SolveTiles T = solve_tiles(nx, ny, W.form);
    nb = T.ntx * T.nty;
    ox = (W.tile % T.ntx) * T.tw;
    oy = (W.tile / T.ntx) * T.th;
    ow = min(T.tw, nx - ox);
    oh = min(T.th, ny - oy);
    round0 = st->rounds[W.form][s];
    most = st->polls;
  }
  if (tid == 0) {
    L.lost = 0;
    L.irregular = 0;
  }
  __syncthreads();

  // The thread's matrix rows, as k_assemble left them, and the start x = b.
  // ALONE: rows tid, tid + NT, ..  Else column `lane` of the tile, whose first
  // own cell is HALO, in the wave's strip of RPT rows; what lies beyond the
  // tile's halo are rows of the grid as well (lanes: rows x = 1 of their own),
  // swept like the others and never looked at, so that no sweep asks.
  double M[RPT][4], D[RPT], R[RPT], b[RPT], x[RPT];
  int at[ALONE ? RPT : 1][4], row[RPT];  // row: the first cell of the grid's row
  const int tx = lane - HALO, ty0 = wv * RPT - HALO;  // within the own cells
  unsigned ci = tid;
  const gdouble* Mp[5];
#pragma unroll
  for (int q = 0; q < 5; ++q) Mp[q] = uniform(G(J.M[s][q]));
  const gdouble* rhs = uniform(system_rhs(J, S));
  double* const buf0 = uniform(J.FX[s][0]);
  double* const buf1 = uniform(J.FX[s][1]);
  if (!ALONE) {
    int c = (ox + tx) % nx, cj = (oy + ty0) % ny;
    ci = c < 0 ? c + nx : c;
    cj = cj < 0 ? cj + ny : cj;
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      row[i] = cj * nx;
      cj = cj + 1 == ny ? 0 : cj + 1;
    }
  }
  const bool held_lane = lane < ow + 2 * HALO, own_lane = tx >= 0 && tx < ow;
  auto held = [&](int i) { return ALONE ? i * NT + tid < n : held_lane; };
  auto own_row = [&](int i) { return ty0 + i >= 0 && ty0 + i < oh; };
  auto own = [&](int i) { return ALONE ? held(i) : own_lane && own_row(i); };
  bool regular = true;
  double bsum = 0.;
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    if (ALONE) {
      const int l = i * NT + tid, cj = l / nx, c = l - cj * nx;
      row[i] = i * NT;
      at[ALONE ? i : 0][0] = (cj == 0 ? ny - 1 : cj - 1) * nx + c;
      at[ALONE ? i : 0][1] = cj * nx + (c == 0 ? nx - 1 : c - 1);
      at[ALONE ? i : 0][2] = cj * nx + (c == nx - 1 ? 0 : c + 1);
      at[ALONE ? i : 0][3] = (cj == ny - 1 ? 0 : cj + 1) * nx + c;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) M[i][q] = 0.;
    D[i] = 1.;
    b[i] = 1.;
  }
  if (held(0)) {
#pragma unroll
    for (int i = 0; i < RPT; ++i)
      if (!ALONE || held(i)) {
#pragma unroll
        for (int q = 0; q < 4; ++q) M[i][q] = (Mp[q] + row[i])[ci];
        D[i] = (Mp[4] + row[i])[ci];
        b[i] = (rhs + row[i])[ci];
      }
  }
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    R[i] = recip_refined(D[i]);
    x[i] = b[i];
    regular = regular & solve_row_regular(M[i], D[i], b[i]);
    if (own(i)) bsum += fabs(0.0 - b[i]);
  }

  // One sweep of every row; returns the thread's part of the own cells'
  // SUM(ABS(x_new - x_old)).  ALONE: from and to in LDS.  Else in the
  // registers: the neighbours to the west and east are the next lanes', those
  // beyond a strip's ends come from the edges of parity `par`, and the new ones
  // go to the other parity unless it is the `last`.  The outermost row of the
  // tile, or lane, takes what it finds, never less than 0: a sweep spoils it.
  auto sweep = [&](auto shrt, const double* from, double* to, int par, bool last) {
    constexpr bool SHORT = decltype(shrt)::value;
    double dsum = 0.;
    if (ALONE) {
#pragma unroll
      for (int i = 0; i < RPT; ++i)
        if (held(i)) {
          const int l = i * NT + tid;
          const int* a = at[ALONE ? i : 0];
          const double c = from[l];
          const double xv = solve_row<SHORT>(M[i], D[i], R[i], b[i], c, from[a[0]], from[a[1]],
                                             from[a[2]], from[a[3]]);
          to[l] = xv;
          dsum += fabs(xv - c);
        }
      __syncthreads();
      return dsum;
    }
    double south = L.t.edge[par][wv ? wv - 1 : 0][1][lane];
    const double north = L.t.edge[par][wv < kSolveWaves - 1 ? wv + 1 : wv][0][lane];
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const double c = x[i];
      const double xv = solve_row<SHORT>(M[i], D[i], R[i], b[i], c, south, dpp<0x138, 0xf>(c),
                                         dpp<0x130, 0xf>(c), i + 1 < RPT ? x[i + 1] : north);
      if (SHORT)
        dsum = fma(fabs(xv - c), own_row(i) ? 1. : 0., dsum);
      else
        dsum += own_row(i) ? fabs(xv - c) : 0.;
      if (!SHORT) __builtin_amdgcn_sched_barrier(0);  // few registers are left at 11 rows
      south = c;
      x[i] = xv;
    }
    if (!last) {
      L.t.edge[par ^ 1][wv][0][lane] = x[0];
      L.t.edge[par ^ 1][wv][1][lane] = x[RPT - 1];
      __syncthreads();
    }
    return own_lane ? dsum : 0.;
  };
  auto publish_edges = [&] {
    L.t.edge[0][wv][0][lane] = x[0];
    L.t.edge[0][wv][1][lane] = x[RPT - 1];
  };

  // certified_continue with the division by n taken to the other side: n tol
  // widened by 2^-50 covers the roundings of both forms, 2^-43 the tags.
  const double tn = E.tol * (double)n, width = fabs(tn) * 0x1p-50;
  const double tn_lo = tn - width, tn_hi = tn + width;
  const double relS = 8.0 * (double)n * 0x1p-53 + (ALONE ? 0. : 0x1p-43);
  auto certified = [&](double sum) {
    const double B = relS * sum;
    if (isnan(sum)) return 0;
    if (isinf(sum) || sum - B > tn_hi) return 1;
    return sum + B <= tn_lo ? 0 : -1;
  };

  if (ALONE) {
#pragma unroll
    for (int i = 0; i < RPT; ++i)
      if (held(i)) L.x[0][i * NT + tid] = x[i];
  } else {
    publish_edges();
  }
  if (!regular) L.irregular = ~0u;
  __syncthreads();
  regular = L.irregular != ~0u;
  double *p0 = L.x[0], *q0 = L.x[1], *q1 = L.x[2];  // ALONE
  int k_sweeps = 0, end = kSolveConverged;
  bool zero = false;
  unsigned t = 0;
  for (;; ++t) {
    double sum[kSolveKinds];
    if (!ALONE) {
#pragma unroll
      for (int i = 0; i < RPT; ++i) L.t.start[i * NT + tid] = x[i];
    }
    static_assert(kSolveWindow == 4, "the sweeps of a window");
    if (regular) {
      constexpr std::true_type shrt;
      sum[0] = sweep(shrt, p0, q0, 0, false);
      sum[1] = sweep(shrt, q0, q1, 1, false);
      sum[2] = sweep(shrt, q1, q0, 0, false);
      sum[3] = sweep(shrt, q0, q1, 1, true);
    } else {
#pragma unroll 1
      for (int k = 0; k < kSolveWindow; ++k) {
        const double v = sweep(std::false_type(), k == 0 ? p0 : k & 1 ? q0 : q1, k & 1 ? q1 : q0,
                               k & 1, k == kSolveWindow - 1);
#pragma unroll
        for (int q = 0; q < kSolveWindow; ++q)
          if (q == k) sum[q] = v;
      }
    }
    sum[kSolveWindow] = bsum;  // used in the first round only
    double* buf = t & 1 ? buf1 : buf0;  // free between an FVTD's update and the next one's face kernels
    if (!ALONE) {
      const bool outer_lane = tx < HALO || tx >= ow - HALO;
#pragma unroll
      for (int i = 0; i < RPT; ++i)
        if (own(i) && (outer_lane || ty0 + i < HALO || ty0 + i >= oh - HALO))
          agent_store(buf + row[i] + ci, x[i]);
    }
#pragma unroll
    for (int q = 0; q < kSolveKinds; ++q) {
      const double w = wave_sum_dpp(sum[q]);
      if ((tid & 63) == 0) L.red[q][tid >> 6] = w;
    }
    if (!ALONE) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    const unsigned tag = (round0 + t + 1u) & 0xffu;
    if (!ALONE) {
      const size_t slot = solve_slot(nx, ny, W.form, s, (round0 + t) & 1u, 0);
      if (tid < kSolveKinds) {
        double v = L.red[tid][0];
        for (int w = 1; w < kSolveWaves; ++w) v += L.red[tid][w];
        __hip_atomic_store(J.slots + slot + (size_t)tid * nb + W.tile,
                           ((unsigned long long)__double_as_longlong(v) & ~0xffull) | tag,
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      // waves 0-3 poll kinds 0, 1 and 4 of block tid (nb <= 256), waves 4-7
      // kinds 2 and 3
      const int half = tid >> 8, blk = tid & 255;
      const int nk = half == 0 && t == 0 ? 3 : 2;
      unsigned long long v[3] = {tag, tag, tag};
      if (blk < nb) {
        int polls = most;
        bool missing;
        do {
          missing = false;
          for (int q = 0; q < nk; ++q) {
            const int kind = q == 2 ? kSolveWindow : 2 * half + q;
            v[q] = __hip_atomic_load(J.slots + slot + (size_t)kind * nb + blk, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
            missing |= (unsigned)(v[q] & 0xffu) != tag;
          }
        } while (missing && --polls > 0);
        if (missing || most <= 0) L.lost = 1;
      }
      for (int q = 0; q < nk; ++q) {
        const double w = wave_sum_dpp(__longlong_as_double((long long)(v[q] & ~0xffull)));
        if ((tid & 63) == 0) L.tot[q == 2 ? kSolveWindow : 2 * half + q][(tid >> 6) & 3] = w;
      }
      __syncthreads();
      if (L.lost) {  // set before the barrier: every thread of the block sees it
        end = kSolveOpen;
        break;
      }
    }
    // the halo of the next window, on its way while the stop rule is applied
    if (!ALONE) {
#pragma unroll
      for (int i = 0; i < RPT; ++i)
        if (!own(i)) x[i] = held(i) && ty0 + i < oh + HALO ? agent_load(buf + row[i] + ci) : 1.;
    }
    // The stop rule (src/jacobi_iteration.f90:63-84), sweep by sweep: the same
    // numbers, and so the same decisions, in every block of the system.  Lane
    // 8q + w of each wave takes part w of sum q; its group of 8 lanes adds
    // them up, and the decisions of all sums come as bits of two ballots.
    double part = 0.;
    if (ALONE) {
      if ((tid & 63) < 8 * kSolveKinds) part = L.red[(tid & 63) >> 3][tid & 7];
    } else {
      if ((tid & 63) < 8 * kSolveKinds && (tid & 7) < 4) part = L.tot[(tid & 63) >> 3][tid & 3];
    }
    part += dpp<0x111, 0xf>(part);
    part += dpp<0x112, 0xf>(part);
    part += dpp<0x114, 0xf>(part);  // lane 8q + 7 (and 8q + 15 of a row) holds its eight
    const int c = certified(part);
    const unsigned long long go = __ballot(c > 0), open = __ballot(c < 0);
    auto decision = [&](int q) {
      const int bit = 8 * q + 7;
      return (int)((go >> bit) & 1u) - (int)((open >> bit) & 1u);
    };
    bool stop = false;
    if (t == 0) {
      const int c0 = decision(kSolveWindow);
      if (c0 < 0) {
        stop = true;
        end = kSolveOpen;
      } else if (!c0 || E.max_iter <= 0) {
        stop = true;
        zero = true;
        end = c0 ? kSolveLimit : kSolveConverged;
      }
    }
    int j = 0;
    for (; j < kSolveWindow && !stop; ++j) {
      ++k_sweeps;
      const int c1 = decision(j);
      stop = true;
      if (c1 < 0)
        end = kSolveOpen;
      else if (c1 == 0)
        end = kSolveConverged;
      else if (k_sweeps >= E.max_iter)
        end = kSolveLimit;
      else if (k_sweeps >= limit)
        end = kSolveOpen;
      else
        stop = false;
    }
    if (stop) {
      // the iterate of the window's sweep j (counted from 1)
      if (end == kSolveOpen || zero) break;
      if (ALONE ? j <= 2 : j < kSolveWindow) {
        if (!ALONE) {
#pragma unroll
          for (int i = 0; i < RPT; ++i) x[i] = L.t.start[i * NT + tid];
          publish_edges();
          __syncthreads();
        }
#pragma unroll 1
        for (int k = 0; k < j; ++k) {
          const double *from = k ? q0 : p0;
          double* to = k ? q1 : q0;
          if (regular)
            sweep(std::true_type(), from, to, k & 1, k == j - 1);
          else
            sweep(std::false_type(), from, to, k & 1, k == j - 1);
        }
      }
      if (ALONE) {
#pragma unroll
        for (int i = 0; i < RPT; ++i)
          if (held(i)) x[i] = (j & 1 ? q0 : q1)[i * NT + tid];
      }
      break;
    }
    unsigned hi = 0;
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      if (ALONE && held(i)) x[i] = q1[i * NT + tid];
      hi = max(hi, (unsigned)__double2hiint(x[i]));
    }
    if (hi >= kSolveStartHi) L.irregular = t + 1;
    if (!ALONE) publish_edges();
    __syncthreads();  // also: the sums have been read
    regular = regular && L.irregular != t + 1;
    double* w = p0;
    p0 = q1;
    q1 = q0;
    q0 = w;
  }
  if (end != kSolveOpen) {
    gdouble* to = uniform(G(J.hres[m]));
#pragma unroll
    for (int i = 0; i < RPT; ++i)
      if (own(i)) (to + row[i])[ci] = zero ? 0. : x[i];
  }
  if (tid == 0) {
    if (!ALONE && L.lost) {
      st->solve_lost = 1;  // keeps the step from being committed
      st->polls = 0;
    }
    if (W.tile == 0) {
      st->ended[first_solve + s] = end;
      st->iters[first_solve + s] = k_sweeps;
      st->ambiguous[first_solve + s] = 0;
      if (!ALONE) st->rounds[W.form][s] = round0 + t + 1u;
    }
  }
}

__global__ __launch_bounds__(kSolveThreads) void k_solve(EngineArgs E, const SolveRef* refs,
                                                         int first, int form, int nb, SysList S,
                                                         int limit, int first_solve) {
  __shared__ SolveShared L;
  SolveRef W;
  if (nb > 0) {
    const int b = first + blockIdx.x;
    W = {E.single, b % nb, (short)(b / nb), (short)form};
  } else {
    W = refs[first + blockIdx.x];
  }
  if (skipped_stage(E, W.job)) return;
  switch (W.form) {
    case 0:
      return solve_block<kSolveRpt[0], false>(L, E, W, S, limit, first_solve);
    case 1:
      return solve_block<kSolveRpt[1], false>(L, E, W, S, limit, first_solve);
    case 2:
      return solve_block<kSolveRpt[2], false>(L, E, W, S, limit, first_solve);
    case 3:
      return solve_block<kSolveRpt[3], false>(L, E, W, S, limit, first_solve);
    case 4:
      return solve_block<kSolveRpt[4], false>(L, E, W, S, limit, first_solve);
    case kSolveForms:
      return solve_block<1, true>(L, E, W, S, limit, first_solve);
    case kSolveForms + 1:
      return solve_block<2, true>(L, E, W, S, limit, first_solve);
    default:
      return solve_block<4, true>(L, E, W, S, limit, first_solve);
  }
}

// min that propagates NaN (the stage check must see a NaN depth)
__device__ __forceinline__ double nan_min(double a, double b) {
  return (a != a || b != b) ? __builtin_nan("") : (a < b ? a : b);
}

__device__ __forceinline__ double block_min_all(double v, double* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = nan_min(v, __shfl_xor(v, off, 64));
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[w] = v;
  __syncthreads();
  double r = nan_min(nan_min(nan_min(red[0], red[1]), red[2]), red[3]);
  __syncthreads();
  return r;
}

// Result of each solve into the node's depth: x[cur], or 0 when no sweep ran
// (src/jacobi_iteration.f90:68, src/timediscretization.f90:898-903).  With
// stage tracking on, each block also leaves the minimum of the depths it
// wrote in the (by now unused) Jacobi partial-sum slot 0.
__global__ __launch_bounds__(256) void k_finalize(EngineArgs E, const TileRef* blocks,
                                                  SysList S) {
  __shared__ double red[4];
  const TileRef T = tile_of(E, blocks, blockIdx.x);
  const JobDev& J = E.jobs[T.job];
  if (skipped(E, T.job)) return;
  const int k = T.tile * kCellBlock + threadIdx.x;
  double mn = __builtin_inf();
  if (k < J.n) {
    for (int s = 0; s < S.count; ++s) {
      const int m = S.m[s];
      const JacState& q = E.status[T.job].st[s];
      const double v = q.zero ? 0. : G(J.xj[m][q.cur])[k];
      G(J.hres[m])[k] = v;
      mn = nan_min(mn, v);
    }
  }
  if (!S.track_min) return;  // uniform
  mn = block_min_all(mn, red);
  if (threadIdx.x == 0) J.part[T.tile] = mn;
}

// One block per job: fold the finalize blocks' minima into the step's
// minimum JobStatus::hmin_step (k_commit merges it into hmin once the step is
// accepted).
__global__ __launch_bounds__(256) void k_stage_min(EngineArgs E, const int* jobs) {
  __shared__ double red[4];
  const int job = job_of(E, jobs, blockIdx.x);
  const JobDev& J = E.jobs[job];
  if (skipped(E, job)) return;
  double mn = __builtin_inf();
  for (int t = threadIdx.x; t < J.nblk; t += blockDim.x) mn = nan_min(mn, J.part[t]);
  mn = block_min_all(mn, red);
  if (threadIdx.x == 0) {
    JobStatus* st = E.status + job;
    st->hmin_step = st->hmin_step_set ? nan_min(st->hmin_step, mn) : mn;
    st->hmin_step_set = 1;
  }
}

// After a correction's Jacobi phase, one thread per job records the solves:
// sweep counts, ambiguous stops and how each ended (a system still running
// needed more sweeps than were launched).
__global__ void k_solve_done(EngineArgs E, const int* jobs, SysList S, int first_solve) {
  if (threadIdx.x != 0) return;
  JobStatus* st = E.status + job_of(E, jobs, blockIdx.x);
  if (E.gated && st->halt) return;
  for (int s = 0; s < S.count; ++s) {
    const JacState& q = st->st[s];
    st->iters[first_solve + s] = q.k;
    st->ambiguous[first_solve + s] = q.ambiguous;
    st->ended[first_solve + s] = q.active    ? kSolveOpen
                                 : q.nonconv ? kSolveLimit
                                             : kSolveConverged;
  }
}

// Whether the step just run is committed: not when the job's batch has already
// stopped, when a solve was left open (U^n is intact and the host redoes the
// step), or when dt is not finite.
__device__ __forceinline__ bool solves_open(const JobStatus* st, int nsolve) {
  int open = st->solve_lost;
  for (int i = 0; i < nsolve; ++i) open |= st->ended[i] == kSolveOpen;
  return open != 0;
}

// U^{n+1} = Ua(MSteps) (src/timediscretization.f90:564,662,762), node
// mf = MSteps - 1 here, of the accepted steps.  TimeStep's partial maxima of
// the next step (next_dt) come from the values on their way, for a pass over
// the state less; small grids save a launch, 2048^2 breaks even (35 + 35 us
// apart, 71 here).
__global__ __launch_bounds__(256) void k_commit(EngineArgs E, const TileRef* blocks, int mf,
                                                int nsolve, int next_dt) {
  const TileRef T = tile_of(E, blocks, blockIdx.x);
  const JobDev& J = E.jobs[T.job];
  const JobStatus* st = E.status + T.job;
  if (st->halt || st->dt_bad || solves_open(st, nsolve)) return;
  const int k = T.tile * kCellBlock + threadIdx.x;
  const bool in = k < J.n;
  double h = 0., hu = 0., hv = 0.;
  if (in) {
    h = G(J.hres[mf])[k];
    hu = G(J.hun[mf])[k];
    hv = G(J.hvn[mf])[k];
    G(J.h)[k] = h;
    G(J.hu)[k] = hu;
    G(J.hv)[k] = hv;
  }
  if (next_dt) timestep_partial(in, J.g, h, hu, hv, J.tspart + 3 * (size_t)T.tile);
}

// ------------------------------------------------------------------------
// The device time loop: up to kMaxBatch steps between host reads.
//
// k_batch_begin starts a batch (one thread per job).  After each step's commit
// k_step_end (one block per job) records a committed step and advances the
// loop: t = t + dt and the output/end test of src/timediscretization.f90:83-94,
// the job's step count and the batch's.  Whatever stops the batch sets halt,
// and every later kernel of the batch skips the job.
// ------------------------------------------------------------------------
__global__ void k_batch_begin(EngineArgs E, const int* jobs, BatchArgs B) {
  if (threadIdx.x != 0) return;
  JobStatus* st = E.status + job_of(E, jobs, blockIdx.x);
  if (B.redo && st->halt != kHaltOverrun) {  // keeps its own stop
    if (!st->halt) st->halt = kHaltMasked;
    return;
  }
  if (st->steps_left == 0) {  // the job has run all its steps
    st->halt = kHaltCount;
    return;
  }
  st->halt = kHaltNone;
  st->solve_lost = 0;
  st->polls = B.polls;
  st->batch_done = 0;
  st->batch_max = B.max_steps;
  if (B.redo) return;  // the redone step keeps the loop's t
  st->loop = B.loop;
  if (B.loop) {
    st->t = B.t;
    st->t_an = B.t_an;
    st->t_end = B.t_end;
  }
}

__device__ __forceinline__ void record_step(JobStatus* st, int nsolve) {
  // lanes 0..12 take a solve each
  const int i = threadIdx.x;
  const bool mine = i < nsolve;
  const int end = mine ? st->ended[i] : kSolveConverged;
  const int amb = mine ? st->ambiguous[i] : 0, sweeps = mine ? st->iters[i] : 0;
  const int done = st->batch_done, bad = st->dt_bad, lost = st->solve_lost;
  const bool open = __any(end == kSolveOpen) || lost;
  const int nonconv = __popcll(__ballot(end == kSolveLimit));
  if (!open && !bad && i < 13) st->rec[done].iters[i] = sweeps;
  int ambiguous = 0;
  if (__any(amb != 0))
    for (int q = 0; q < 13; ++q) ambiguous += __shfl(amb, q, 64);
  if (i != 0) return;
  if (open || bad) {
    st->halt = open ? kHaltOverrun : kHaltDtBad;
    st->hmin_step_set = 0;  // a redone attempt's stages start a new minimum
    return;
  }
  StepRec& r = st->rec[done];
  r.dt = st->dt;
  r.nonconv = nonconv;
  r.ambiguous = ambiguous;
  st->batch_done = done + 1;
  if (st->hmin_step_set) {  // the accepted step's stage minimum joins the record
    st->hmin = st->hmin_set ? nan_min(st->hmin, st->hmin_step) : st->hmin_step;
    st->hmin_set = 1;
    st->hmin_step_set = 0;
  }
  int halt = kHaltNone;
  if (st->loop) {
    const double t = st->t + st->dt;
    st->t = t;
    if (fabs(st->t_an - t) < 1.0E-10 || fabs(t - st->t_end) < 1.0E-10) halt = kHaltReached;
  }
  const int left = st->steps_left;  // < 0: none
  if (left > 0) {
    st->steps_left = left - 1;
    if (left == 1 && !halt) halt = kHaltCount;
  }
  if (!halt && done + 1 >= st->batch_max) halt = kHaltBatch;
  if (halt) st->halt = halt;
}

// TimeStep of the job's state from the partial maxima, and the time loop's
// dt = MIN(MIN(dt_min, tAnalyze-t), MIN(dt_min, tEnd-t))
// (src/timediscretization.f90:58-59) when the device runs the loop.
template <int NT>
__device__ __forceinline__ void next_step_dt(const JobDev& J, JobStatus* st, int nparts) {
  const gdouble *h = G(J.h), *hu = G(J.hu), *hv = G(J.hv);
  double ts, LX, LY;
  timestep_final<NT>(
      J.tspart, nparts, J.n,
      [&](int k, double& a, double& b, double& c) {
        a = h[k];
        b = hu[k];
        c = hv[k];
      },
      J.g, J.dx, J.dy, J.cfl, ts, LX, LY);
  if (threadIdx.x != 0) return;
  st->dt_min = ts;
  const double dt =
      st->loop ? min_r(min_r(ts, st->t_an - st->t), min_r(ts, st->t_end - st->t)) : ts;
  st->dt = dt;
  st->lmx = LX;
  st->lmy = LY;
  st->dt_bad = isfinite(dt) ? 0 : 1;
}

// The step's record and, when the batch goes on, the next step's dt: one launch
// where the record, TimeStep's maxima and their fold were three (of 4.4 us each
// at 32^2).  mf >= 0: the commit of node mf too, by the job's one block.
__global__ __launch_bounds__(1024) void k_step_end(EngineArgs E, const int* jobs, int mf,
                                                   int nsolve, int next_dt) {
  constexpr int NT = 1024;
  const int job = job_of(E, jobs, blockIdx.x);
  const JobDev& J = E.jobs[job];
  JobStatus* st = E.status + job;
  if (st->halt) return;
  const bool committed = mf < 0 || (!st->dt_bad && !solves_open(st, nsolve));
  if (mf >= 0 && committed) {
    // each 256-thread quarter stands for a block of k_commit
    for (int k0 = 0; k0 < J.n; k0 += NT) {
      const int k = k0 + threadIdx.x;
      const bool in = k < J.n;
      double h = 0., hu = 0., hv = 0.;
      if (in) {
        h = G(J.hres[mf])[k];
        hu = G(J.hun[mf])[k];
        hv = G(J.hvn[mf])[k];
        G(J.h)[k] = h;
        G(J.hu)[k] = hu;
        G(J.hv)[k] = hv;
      }
      if (next_dt) timestep_wave(in, J.g, h, hu, hv, J.tspart + 3 * (k >> 6));
    }
  }
  __shared__ int go_on;
  __syncthreads();  // the maxima are written, and every thread has read the status
  if (threadIdx.x < 64) {
    record_step(st, nsolve);
    if (threadIdx.x == 0) go_on = !st->halt;
  }
  __syncthreads();
  if (next_dt && go_on) next_step_dt<NT>(J, st, mf >= 0 ? (J.n + 63) / 64 : J.nblk);
}

__global__ void k_set_steps_left(JobStatus* st, int steps_left) {
  if (threadIdx.x == 0 && blockIdx.x == 0) st->steps_left = steps_left;
}

// The reference's view of the depths in the two-node schemes.
// MODIFIED_PATANKAR_MATRIX_INVERSION declares hp(MSteps, nx, ny)
// (src/timediscretization.f90:783) and receives Up(:,1,1:nx,1:ny), whose
// first extent is 4 (src/finitevolume.f90:161), so hp is sequence associated:
// hp(m, cell) is element L = (m-1) + 2*cell of Up(1:4, 1, cells) in array
// element order, i.e. node L % 4 of cell L / 4 (cell = (i-1) + nx*(j-1), our
// k).  Nodes 3 and 4 are never written by these schemes and hold 0
// (src/finitevolume.f90:207-208).  So, with m = 2 the node solved:
//   hp(2, k) = k even ? Up(2)[k/2] : 0       -> hres[3]
//   rhs(k)  = hp(1, k) = k even ? h^n[k/2] : 0 -> hres[2]
// where Up(2) is h^n in the first correction (from_un) and node 1's depth
// after it.  hres[2] and hres[3] are free: only node 1 is solved.
__global__ __launch_bounds__(256) void k_hp_view(EngineArgs E, const TileRef* blocks,
                                                 int from_un) {
  const TileRef T = tile_of(E, blocks, blockIdx.x);
  const JobDev& J = E.jobs[T.job];
  if (skipped_stage(E, T.job)) return;
  const int k = T.tile * kCellBlock + threadIdx.x;
  if (k >= J.n) return;
  const gdouble* up2 = G(from_un ? J.h : J.hres[1]);
  const bool odd = k & 1;
  const int c = k >> 1;
  G(J.hres[3])[k] = odd ? 0. : up2[c];
  G(J.hres[2])[k] = odd ? 0. : G(J.h)[c];
}

// A stage combination of an explicit scheme (CombOp, mode 0/1/2), for the
// three variables of every cell.  Reads only slots other than op.out.
__device__ __forceinline__ const gdouble* state_var(const JobDev& J, int v, int s) {
  return G(v == 0 ? J.sh[s] : v == 1 ? J.shu[s] : J.shv[s]);
}
__device__ __forceinline__ const gdouble* deriv_var(const JobDev& J, int v, int r) {
  return G(v == 0 ? J.d1[r] : v == 1 ? J.d2[r] : J.d3[r]);
}

// Every source value is loaded once per variable (fully unrolled over
// kMaxTerms, guarded by nterm, so the values stay in registers) and serves
// each of the op.nout outputs, which differ only in their weights.
//
// FRESH: op.nfresh derivatives are still the fluxes of the FVTD before, in
// their scratch slots, with the sources in d2, d3; they are taken from there
// (update_cell's arithmetic) and stored only where a later stage reads them
// again.  That spares the update's launch and its pass over memory: per stage
// 64^2 7.7 -> 5.8 us (RK65), 300x417 11.0 -> 8.3 (SSPRK4), 1000x700 55 -> 38
// (DeC5, three nodes), 1500x1400 87 -> 68 (RK65).  Bound by latency on small
// grids, by memory on large ones, where the blocks in runs per XCD share the
// rows' y fluxes (1000x700: 45 -> 38).
template <bool FRESH>
__global__ __launch_bounds__(256) void k_combine(EngineArgs E, const TileRef* blocks, int nblocks,
                                                 CombOp op) {
  const int place = FRESH ? xcd_chunk(blockIdx.x, nblocks) : blockIdx.x;
  if (FRESH && place >= nblocks) return;
  const TileRef T = tile_of(E, blocks, place);
  const JobDev& J = E.jobs[T.job];
  if (skipped_stage(E, T.job)) return;
  const int k0 = T.tile * kCellBlock, k = k0 + threadIdx.x;
  if (k >= J.n) return;
  const double dt = E.status[T.job].dt;
  // The loads of a phase before any use or store: a chain of them, pointers from
  // the job's descriptor first, is most of what small grids wait for.
  double base[3], x[3][kMaxTerms];
#pragma unroll
  for (int t = 0; t < kMaxTerms; ++t)
    if (t < op.nterm && !(FRESH && op.fresh[t] >= 0)) {
#pragma unroll
      for (int v = 0; v < 3; ++v)
        x[v][t] = op.deriv[t] ? deriv_var(J, v, op.src[t])[k] : state_var(J, v, op.src[t])[k];
    }
#pragma unroll
  for (int v = 0; v < 3; ++v) base[v] = op.mode == 0 ? 0. : state_var(J, v, op.base)[k];
  if (FRESH) {
    int ci, cj;
    cell_ij(k0 % J.nx, k0 / J.nx, threadIdx.x, J.nx, ci, cj);
    const size_t fw = (size_t)cj * (J.nx + 1) + ci, fe = fw + 1;  // x faces
    const size_t gs = k, gn = gs + J.nx;                          // y faces
    const OverDx over(J);
    double ut[kSlots][3];
#pragma unroll
    for (int q = 0; q < kSlots; ++q)
      if (q < op.nfresh) {
        const int sl = op.fslot[q], to = op.fsrc[q];
        double a[3], b[3], qa[3], qb[3], S[3] = {0., 0., 0.};
        Numerators num{over.shared};
#pragma unroll
        for (int v = 0; v < 3; ++v) {
          const double fxe = G(J.FX[sl][v])[fe], fxw = G(J.FX[sl][v])[fw];
          const double fyn = G(J.FY[sl][v])[gn], fys = G(J.FY[sl][v])[gs];
          if (v > 0 && J.bathy)
            S[v] = deriv_var(J, v, to)[k];
          else if (v > 0 && J.wb)
            S[v] = S[v] - G(v == 1 ? J.SWB2 : J.SWB3)[k];
          a[v] = fxe - fxw;
          b[v] = fyn - fys;
        }
#pragma unroll
        for (int v = 0; v < 3; ++v) {
          qa[v] = div_by(num(a[v]), over.dx, over.rdx);
          qb[v] = div_by(num(b[v]), over.dy, over.rdy);
        }
        if (!num.ok) {
#pragma unroll
          for (int v = 0; v < 3; ++v) {
            qa[v] = over.x(a[v]);
            qb[v] = over.y(b[v]);
          }
        }
        // the source is never -0, so the sign of a zero quotient has no effect
#pragma unroll
        for (int v = 0; v < 3; ++v) ut[q][v] = S[v] - qa[v] - qb[v];
        if (op.fstore[q]) {
          G(J.d1[to])[k] = ut[q][0];
          G(J.d2[to])[k] = ut[q][1];
          G(J.d3[to])[k] = ut[q][2];
        }
        // a derivative at a time: the loads of all three take 152 registers
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
    for (int t = 0; t < kMaxTerms; ++t)
#pragma unroll
      for (int v = 0; v < 3; ++v)
#pragma unroll
        for (int q = 0; q < kSlots; ++q)
          if (t < op.nterm && op.fresh[t] == q) x[v][t] = ut[q][v];
  }
#pragma unroll
  for (int v = 0; v < 3; ++v) {
#pragma unroll
    for (int o = 0; o < kMaxOut; ++o) {
      if (o >= op.nout) break;
      const double* c = op.c[o];
      double acc = 0.;
      if (op.mode == 0) {
#pragma unroll
        for (int t = 0; t < kMaxTerms; ++t)
          if (t < op.nterm) {
            const double term = op.deriv[t] ? (c[t] * x[v][t]) * dt : c[t] * x[v][t];
            acc = t == 0 ? term : acc + term;
          }
      } else if (op.mode == 1) {
        double sum = 0.;
#pragma unroll
        for (int t = 0; t < kMaxTerms; ++t)
          if (t < op.nterm) {
            const double term = c[t] * x[v][t];
            sum = t == 0 ? term : sum + term;
          }
        acc = base[v] + sum * dt;
      } else {
        acc = base[v];
#pragma unroll
        for (int t = 0; t < kMaxTerms; ++t)
          if (t < op.nterm) acc = acc + (dt * c[t]) * x[v][t];
      }
      const int out = op.out[o];
      G(v == 0 ? J.sh[out] : v == 1 ? J.shu[out] : J.shv[out])[k] = acc;
    }
  }
}

// FXWB/FYWB from the slot scratch after the well-balanced FVTD.  The job's
// cell blocks cover n indices; the loop also covers the nx (ny) extra faces.
__global__ __launch_bounds__(256) void k_copy_wb(EngineArgs E, const TileRef* blocks, int slot) {
  const TileRef T = tile_of(E, blocks, blockIdx.x);
  const JobDev& J = E.jobs[T.job];
  const int nfx = (J.nx + 1) * J.ny, nfy = J.nx * (J.ny + 1);
  for (int k = T.tile * kCellBlock + threadIdx.x; k < nfx || k < nfy;
       k += J.nblk * kCellBlock) {
    for (int v = 0; v < 3; ++v) {
      if (k < nfx) G(J.FXWB[v])[k] = G(J.FX[slot][v])[k];
      if (k < nfy) G(J.FYWB[v])[k] = G(J.FY[slot][v])[k];
    }
  }
}

// ------------------------------------------------------------------------
// TimeStep (src/equation.f90:791-837): per-block maxima of the wave speeds,
// then one block per job folds them (swm_timestep.hpp) and applies the time
// loop's clipping.
// ------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_timestep(EngineArgs E, const TileRef* blocks) {
  const TileRef T = tile_of(E, blocks, blockIdx.x);
  const JobDev& J = E.jobs[T.job];
  if (skipped(E, T.job)) return;
  const int k = T.tile * kCellBlock + threadIdx.x;
  const bool in = k < J.n;
  timestep_partial(in, J.g, in ? G(J.h)[k] : 0., in ? G(J.hu)[k] : 0., in ? G(J.hv)[k] : 0.,
                   J.tspart + 3 * (size_t)T.tile);
}

template <int NT>
__global__ __launch_bounds__(NT) void k_timestep_final(EngineArgs E, const int* jobs) {
  const int job = job_of(E, jobs, blockIdx.x);
  if (skipped(E, job)) return;
  next_step_dt<NT>(E.jobs[job], E.status + job, E.jobs[job].nblk);
}

// ------------------------------------------------------------------------
// Layout conversion between the reference's U(1:3, ...) and device SoA.
// ghost = 3: the source is U(1:3, -2:nx+3, -2:ny+3) including ghosts.
// ------------------------------------------------------------------------
__global__ void k_aos_to_soa(int nx, int ny, int ghost, const double* aos, double* h, double* hu,
                             double* hv) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nx * ny) return;
  int i = k % nx, j = k / nx;
  size_t src = 3 * ((size_t)(j + ghost) * (nx + 2 * ghost) + (i + ghost));
  h[k] = aos[src];
  hu[k] = aos[src + 1];
  hv[k] = aos[src + 2];
}

__global__ void k_soa_to_aos(int nx, int ny, const double* h, const double* hu, const double* hv,
                             double* aos) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nx * ny) return;
  aos[3 * (size_t)k] = h[k];
  aos[3 * (size_t)k + 1] = hu[k];
  aos[3 * (size_t)k + 2] = hv[k];
}

// A chunk of a state to the pinned ring, or (UP) from it.  The ring's side goes by
// system-scope accesses, which no cache of the device keeps.  Bound by the bus: 101 MB
// in chunks of 1 MB 2.4 ms either way, with 128 and 256 blocks the same.
constexpr int kRingCopyBlocks = 64;
template <bool UP>
__global__ __launch_bounds__(256) void k_ring_copy(const double* from, double* to, size_t n) {
  const size_t step = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += 4 * step) {
    double v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (i + u * step >= n) continue;
      v[u] = UP ? __hip_atomic_load(from + i + u * step, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_SYSTEM)
                : from[i + u * step];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (i + u * step >= n) continue;
      if (UP)
        to[i + u * step] = v[u];
      else
        __hip_atomic_store(to + i + u * step, v[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

__global__ void k_divsqrt(int n, const double* a, const double* b, double* q, double* r) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  q[k] = a[k] / b[k];
  r[k] = sqrt(a[k]);
}

// a/b through the shared-reciprocal sequence (recip_refined + div_by),
// without the range check, for comparison with '/'.
__global__ void k_shared_div(int n, const double* a, const double* b, double* q) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  q[k] = div_by(a[k], b[k], recip_refined(b[k]));
}

// WENO5 first sweep (out: wm, wp) and second sweep (out: 4 Gauss-point
// values) of n five-point stencils q[5*i .. 5*i+4], as the kernels compute them.
__global__ void k_weno5(int n, const double* q, double* first, double* second) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const double* s = q + 5 * (size_t)k;
  double wm, wp, w[4];
  weno5_first(s[0], s[1], s[2], s[3], s[4], wm, wp);
  weno5_second(s[0], s[1], s[2], s[3], s[4], w);
  first[2 * (size_t)k] = wm;
  first[2 * (size_t)k + 1] = wp;
  for (int g = 0; g < 4; ++g) second[4 * (size_t)k + g] = w[g];
}

// ------------------------------------------------------------------------
// The state the reference's output writer prints: WriteSolutionToDisk
// (src/output.f90:79) writes the module array V, which the last FVTD of the
// step filled from its input -- for mPDeC5 the fourth DeC node after the
// fourth correction (src/timediscretization.f90:548-556), not U^{n+1}.  A copy
// of that node's state for the jobs that asked for it (vout != null).
// ------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_keep_state(EngineArgs E, const TileRef* blocks, int m) {
  const TileRef T = tile_of(E, blocks, blockIdx.x);
  const JobDev& J = E.jobs[T.job];
  if (skipped(E, T.job)) return;
  if (!J.vout) return;
  const int k = T.tile * kCellBlock + threadIdx.x;
  if (k >= J.n) return;
  const gdouble *h, *hu, *hv;
  node_state(J, m, h, hu, hv);
  gdouble* o = G(J.vout);
  o[k] = h[k];
  o[J.n + k] = hu[k];
  o[2 * (size_t)J.n + k] = hv[k];
}

// ------------------------------------------------------------------------
// launch wrappers
// ------------------------------------------------------------------------
static inline unsigned cdiv(long a, long b) { return (unsigned)((a + b - 1) / b); }

void launch_fvtd(const EngineArgs& E, int shape, const TileRef* xt, int nxt, const TileRef* yt,
                 int nyt, const TileRef* st, int nst, const NodeList& L, hipStream_t s) {
  static_assert(kNumShapes == 2 && kAllShapes == 3 && kShapes[0].xw == 16 && kShapes[0].xh == 16 &&
                    kShapes[0].yw == 16 && kShapes[0].yh == 16 && kShapes[0].sw == 16 &&
                    kShapes[0].sh == 16 && kShapes[1].xw == 32 && kShapes[1].xh == 16 &&
                    kShapes[1].yw == 16 && kShapes[1].yh == 32 && kShapes[1].sw == 32 &&
                    kShapes[1].sh == 16,
                "the instantiations below follow kShapes");
  const FvtdTiles T = {xt, yt, st, nxt, nyt, nst};
  const unsigned groups = cdiv((long)(nxt + nyt) * L.count, 8) + cdiv(nst, 8) * L.count;
  if (!groups) return;
  if (shape == kSplitShape)
    hipLaunchKernelGGL((k_fvtd<16, 8, 8, 16, 16, 16, true>), dim3(groups * 8), dim3(256), 0, s, E,
                       T, L);
  else if (shape == 1)
    hipLaunchKernelGGL((k_fvtd<32, 16, 16, 32, 32, 16>), dim3(groups * 8), dim3(512), 0, s, E, T,
                       L);
  else
    hipLaunchKernelGGL((k_fvtd<16, 16, 16, 16, 16, 16>), dim3(groups * 8), dim3(256), 0, s, E, T,
                       L);
}

void launch_fvtd_source_update(const EngineArgs& E, const TileRef* ct, int nct, const NodeList& L,
                               hipStream_t s) {
  if (nct)
    hipLaunchKernelGGL(k_fvtd_source_update, dim3(cdiv(nct, 8) * 8 * L.count), dim3(256), 0, s, E,
                       ct, nct, L);
}

void launch_fvtd_update(const EngineArgs& E, const TileRef* cb, int ncb, const NodeList& L,
                        hipStream_t s) {
  if (ncb)
    hipLaunchKernelGGL(k_fvtd_update, dim3(ncb, L.count), dim3(256), 0, s, E, cb, L);
}

void launch_keep_state(const EngineArgs& E, const TileRef* cb, int ncb, int m, hipStream_t s) {
  if (ncb) hipLaunchKernelGGL(k_keep_state, dim3(ncb), dim3(256), 0, s, E, cb, m);
}

template <bool FIRST>
void assemble(dim3 grid, const EngineArgs& E, const TileRef* cb, int nb, const SysList& S,
              hipStream_t s) {
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, E, cb, nb, S); };
  if (S.nr == 2)
    S.fresh == 2 ? go(k_assemble<2, FIRST, 2>)
                 : S.fresh ? go(k_assemble<2, FIRST, 1>) : go(k_assemble<2, FIRST>);
  else
    S.fresh == 2 ? go(k_assemble<4, FIRST, 2>)
                 : S.fresh ? go(k_assemble<4, FIRST, 1>) : go(k_assemble<4, FIRST>);
}

void launch_assemble(const EngineArgs& E, const TileRef* cb, int ncb, const int* jl, int njobs,
                     const SysList& S, hipStream_t s) {
  if (!ncb) return;
  const int nb = cdiv(ncb, sum_blocks(E, ncb));  // one job: ncb is its nblk
  assemble<true>(dim3(xcd_blocks(nb)), E, cb, nb, S, s);
  hipLaunchKernelGGL(k_decide<true>, dim3(njobs), dim3(256), 0, s, E, jl, S);
}

void launch_hp_view(const EngineArgs& E, const TileRef* cb, int ncb, int from_un, hipStream_t s) {
  if (ncb) hipLaunchKernelGGL(k_hp_view, dim3(ncb), dim3(256), 0, s, E, cb, from_un);
}

void launch_combine(const EngineArgs& E, const TileRef* cb, int ncb, const CombOp& op,
                    hipStream_t s) {
  if (!ncb) return;
  if (op.nfresh)
    hipLaunchKernelGGL(k_combine<true>, dim3(xcd_blocks(ncb)), dim3(256), 0, s, E, cb, ncb, op);
  else
    hipLaunchKernelGGL(k_combine<false>, dim3(ncb), dim3(256), 0, s, E, cb, ncb, op);
}

void launch_sweep(const EngineArgs& E, const TileRef* cb, int ncb, const int* jl, int njobs,
                  const SysList& S, hipStream_t s) {
  if (!ncb) return;
  hipLaunchKernelGGL(k_sweep, dim3(ncb), dim3(256), 0, s, E, cb, S);
  hipLaunchKernelGGL(k_decide<false>, dim3(njobs), dim3(256), 0, s, E, jl, S);
}

// A block of k_assemble holds 33 KB of LDS, so 1024 run at once; below that
// the systems of a cell get blocks of their own (32^2: 12 -> 6 us), from
// there on one block shares the face fluxes between them.
void launch_assemble_matrix(const EngineArgs& E, const TileRef* cb, int ncb, const SysList& S,
                            hipStream_t s) {
  if (!ncb) return;
  assemble<false>(dim3(xcd_blocks(ncb), ncb < 1024 ? S.count : 1), E, cb, ncb, S, s);
}

void launch_solve(const EngineArgs& E, const SolveRef* refs, int first, int nblk, int form, int nb,
                  const SysList& S, int limit, int first_solve, hipStream_t s) {
  if (nblk)
    hipLaunchKernelGGL(k_solve, dim3(nblk), dim3(kSolveThreads), 0, s, E, refs, first, form, nb, S,
                       limit, first_solve);
}

void launch_finalize(const EngineArgs& E, const TileRef* cb, int ncb, const int* jl, int njobs,
                     const SysList& S, hipStream_t s) {
  if (!ncb) return;
  hipLaunchKernelGGL(k_finalize, dim3(ncb), dim3(256), 0, s, E, cb, S);
  if (S.track_min) hipLaunchKernelGGL(k_stage_min, dim3(njobs), dim3(256), 0, s, E, jl);
}

void launch_timestep(const EngineArgs& E, const TileRef* cb, int ncb, const int* jl, int njobs,
                     hipStream_t s) {
  if (!ncb) return;
  hipLaunchKernelGGL(k_timestep, dim3(ncb), dim3(256), 0, s, E, cb);
  // 256 threads up to 2048 partial maxima a job, on average: they start sooner
  // (32^2 3.2 us against 4.6, 512^2 3.8 / 4.8, 700^2 4.5 / 4.8); more of them read
  // faster with 1024 (1024^2 6.6 / 5.1, 2048^2 20.6 / 9.4)
  if (ncb <= 2048L * njobs)
    hipLaunchKernelGGL(k_timestep_final<256>, dim3(njobs), dim3(256), 0, s, E, jl);
  else
    hipLaunchKernelGGL(k_timestep_final<1024>, dim3(njobs), dim3(1024), 0, s, E, jl);
}

void launch_commit(const EngineArgs& E, const TileRef* cb, int ncb, int final_node, int nsolve,
                   int next_dt, hipStream_t s) {
  if (ncb)
    hipLaunchKernelGGL(k_commit, dim3(ncb), dim3(256), 0, s, E, cb, final_node, nsolve, next_dt);
}

void launch_step_end(const EngineArgs& E, const int* jl, int njobs, int final_node, int nsolve,
                     int next_dt, hipStream_t s) {
  if (njobs)
    hipLaunchKernelGGL(k_step_end, dim3(njobs), dim3(1024), 0, s, E, jl, final_node, nsolve,
                       next_dt);
}

void launch_batch_begin(const EngineArgs& E, const int* jl, int njobs, const BatchArgs& B,
                        hipStream_t s) {
  if (njobs) hipLaunchKernelGGL(k_batch_begin, dim3(njobs), dim3(64), 0, s, E, jl, B);
}

void launch_set_steps_left(JobStatus* st, int steps_left, hipStream_t s) {
  hipLaunchKernelGGL(k_set_steps_left, dim3(1), dim3(64), 0, s, st, steps_left);
}

void launch_solve_done(const EngineArgs& E, const int* jl, int njobs, const SysList& S,
                       int first_solve, hipStream_t s) {
  if (njobs) hipLaunchKernelGGL(k_solve_done, dim3(njobs), dim3(64), 0, s, E, jl, S, first_solve);
}

void launch_copy_wb(const EngineArgs& E, const TileRef* cb, int ncb, int slot, hipStream_t s) {
  if (ncb) hipLaunchKernelGGL(k_copy_wb, dim3(ncb), dim3(256), 0, s, E, cb, slot);
}

void launch_aos_to_soa(int nx, int ny, int ghost, const double* aos, double* h, double* hu,
                       double* hv, hipStream_t s) {
  hipLaunchKernelGGL(k_aos_to_soa, dim3(cdiv((long)nx * ny, 256)), dim3(256), 0, s, nx, ny,
                     ghost, aos, h, hu, hv);
}

void launch_soa_to_aos(int nx, int ny, const double* h, const double* hu, const double* hv,
                       double* aos, hipStream_t s) {
  hipLaunchKernelGGL(k_soa_to_aos, dim3(cdiv((long)nx * ny, 256)), dim3(256), 0, s, nx, ny, h,
                     hu, hv, aos);
}

void launch_ring_copy(const double* from, double* to, size_t n, bool up, hipStream_t s) {
  const dim3 grid(kRingCopyBlocks), block(256);
  if (up)
    hipLaunchKernelGGL((k_ring_copy<true>), grid, block, 0, s, from, to, n);
  else
    hipLaunchKernelGGL((k_ring_copy<false>), grid, block, 0, s, from, to, n);
}

void launch_divsqrt(int n, const double* a, const double* b, double* q, double* r,
                    hipStream_t s) {
  hipLaunchKernelGGL(k_divsqrt, dim3(cdiv(n, 256)), dim3(256), 0, s, n, a, b, q, r);
}

void launch_weno5(int n, const double* q, double* first, double* second, hipStream_t s) {
  hipLaunchKernelGGL(k_weno5, dim3(cdiv(n, 256)), dim3(256), 0, s, n, q, first, second);
}

void launch_shared_div(int n, const double* a, const double* b, double* q, hipStream_t s) {
  hipLaunchKernelGGL(k_shared_div, dim3(cdiv(n, 256)), dim3(256), 0, s, n, a, b, q);
}

}  // namespace swm
