// k_solve.hip -- K5: the implicit viscous solve of one RK3 substep
// (linsolve, linsolve_blocking.inc:3-107).  Grids whose columns fit in LDS
// (ny <= 130) take k_solve_lds and k_mean; the others three kernels:
//
//   k_solve_ve (k_solve_ve_wide on wide grids) : one lane per (pair, system, real/imaginary part); system 0 =
//                eta, 1 = v.  The pairs (kx, kz) and (kx, -kz) have the same
//                k^2, hence the same matrix: their four lanes (sign x part)
//                sit side by side and share one row of stored lower factors.
//                Builds the pentadiagonal rows lambda*D - nu*L
//                of etamat / D2vmat, folds the wall conditions into rows 1,2
//                and ny-2,ny-1 (applybc_0 / applybc_n, dnsdata.f90:458-472),
//                factorises bottom-up with reciprocal pivots fused with the
//                backward sweep (LU5decompStep + LeftLU5divStep1,
//                rbparmat_blocking.f90:20-77), then runs the forward sweep
//                (LeftLU5divStep2, :82-100) and recovers wall and ghost values
//                (linsolve_blocking.inc:50-61).  The matrices are real, so the
//                real and imaginary parts of a right-hand side are independent
//                recurrences on adjacent lanes.  All four lanes of a group
//                store the same lower factors, so each reads back only what
//                it wrote itself.
//                The spare pair slot npair (plane padding) solves the
//                unit-forcing response ucor: the (0,0) eta matrix with
//                right-hand side 1 and homogeneous walls (:65-76).
//   k_mean     : the (0,0) mode: u/w split, flow rates by the three-point
//                integral (yintegr, dnsdata.f90:312-324), constant-flow
//                correction or CPI pressure gradient (linsolve_blocking.inc:62-97).
//   k_uw       : every other pair, one lane per real/imaginary part: dv/dy by
//                the compact first derivative (COMPLEXderiv + LeftLU5divStep2
//                with D0, dnsdata.f90:337-373) and u = (i kx v' - i kz eta)/k^2,
//                w = (i kz v' + i kx eta)/k^2 (linsolve_blocking.inc:99-103).
//
// The factorisation order of k_solve_ve and k_uw (bottom-up UL, no pivoting) is
// the reference's; k_solve_lds eliminates from both walls.  FP64 results agree
// to rounding either way.
//
// Every sweep loads PF rows ahead into a register ring.  The ring loads are
// unconditional (row indices clamped into the column), so no ring register
// is ever the merge of a loaded and an old value: such a merge makes the
// compiler wait for the load at once and serialises the sweep on memory
// latency.  Full groups of PF rows run in the main loop, the last partial
// group from the ring alone.
#include <type_traits>

#include "chan_internal.hpp"

namespace chan {

constexpr int PF = 4;  // rows of software prefetch in the sequential sweeps

// Block b of a grid of nb = 8m blocks solves column block (b % 8) m + b / 8:
// round-robin dispatch then gives each XCD a contiguous run of column blocks,
// so the cache lines that neighbouring blocks share (a block's pair range
// starts and ends inside a line) stay in one L2.  2% on k_solve_ve at
// 191x384x189; the extra blocks of the rounded grid exit at once.
__device__ __forceinline__ int xcd_block(int b, int nb) {
  return (b & 7) * (nb >> 3) + (b >> 3);
}
// elements per row of the lower factors: a group each, and ucor's
__host__ __device__ __forceinline__ size_t group_stride(int ngrp) { return ((size_t)ngrp + 1 + 63) / 64 * 64; }
static unsigned xcd_grid(size_t lanes) {
  return (unsigned)(((lanes + 255) / 256 + 7) / 8 * 8);
}

// One band: the pentadiagonal rows of etamat (SYS 0) or D2vmat (SYS 1) of a
// wavenumber pair, with the wall conditions folded in: lambda D0 - SQ for eta,
// lambda (D2 - k2 D0) - OS for v, each inner row's entry rounded as the reference forms
// it (the v band's condition number reaches 1e6, so other groupings of the same
// sums move the solution by 1e-12 of it); the wall columns are folded in by ratios
// formed beforehand.
struct Band {
  const double *bc0, *bc0m1, *bcn, *bcnp1;  // wall rows
  const WallRatios *q;                      // their ratios
  double lambda, ni, k2, eta0, etan;
  int ny;

  __device__ __forceinline__ Band(const SolveArgs &a, int sys, double k2, double eta0, double etan)
      : bc0(a.bc[sys ? BC_V0 : BC_ETA0]), bc0m1(a.bc[sys ? BC_V0M1 : BC_ETA0M1]), bcn(a.bc[sys ? BC_VN : BC_ETAN]),
        bcnp1(a.bc[sys ? BC_VNP1 : BC_ETANP1]), q(&a.wall[sys]), lambda(a.lambda), ni(a.ni), k2(k2), eta0(eta0),
        etan(etan), ny(a.g.ny) {}
};

// 1/a from the hardware's approximation and two Newton steps: the correctly rounded
// quotient but where the mantissa of a is one of the six largest (then one unit off in the
// last place; compared with the division for 5e10 arguments), in half the dependent
// operations of the division, which is the longest link of the bottom-up sweep's chain.
__device__ __forceinline__ double recip(double a) {
  double r = __builtin_amdgcn_rcp(a);
  r = fma(fma(-a, r, 1.0), r, r);
  return fma(fma(-a, r, 1.0), r, r);
}

// The bottom-up sweep: factorises row iy against the rows iy+1, iy+2 done
// before it, advances the backward substitution (x1) and returns the row's two
// lower factors.
template <int SYS>
struct UpState {
  double l1m2 = 0.0, l1m1 = 0.0, l2m2 = 0.0, l2m1 = 0.0;  // lower factors of rows iy+1, iy+2
  double x1 = 0.0, x2 = 0.0;

  // The row of A with right-hand side b against the two rows done before it:
  // factors it (A[0], A[1] become the lower factors) and advances x1.
  __device__ __forceinline__ void step(double (&A)[5], double b) {
    const double p2 = A[4];
    A[3] = A[3] - p2 * l2m1;
    A[2] = A[2] - p2 * l2m2;
    const double p1 = A[3];
    A[2] = A[2] - p1 * l1m1;
    A[1] = A[1] - p1 * l1m2;
    const double r = recip(A[2]);
    A[0] = A[0] * r;
    A[1] = A[1] * r;
    const double xi = (b - (p1 * x1 + p2 * x2)) * r;
    l2m2 = l1m2;
    l2m1 = l1m1;
    l1m2 = A[0];
    l1m1 = A[1];
    x2 = x1;
    x1 = xi;
  }

  // d: the row's stencils d0, d2 and, for v, d4
  __device__ __forceinline__ static void coefficients(const Band &B, const double (&d)[SYS ? 15 : 10], double (&A)[5]) {
#pragma unroll
    for (int j = 0; j < 5; j++) {
      const double d0 = d[j], d2 = d[5 + j];
      if constexpr (SYS) {
        const double os = B.ni * (d[10 + j] - 2.0 * B.k2 * d2 + B.k2 * B.k2 * d0);
        A[j] = B.lambda * (d2 - B.k2 * d0) - os;
      } else {
        const double sq = B.ni * (d2 - B.k2 * d0);
        A[j] = B.lambda * d0 - sq;
      }
    }
  }

  // WALL: rows 1, 2, ny-2 and ny-1, whose wall columns are folded (applybc_0 /
  // applybc_n); they run from a loop of their own, so that the unrolled inner
  // rows stay short.
  template <bool WALL>
  __device__ __forceinline__ double2 row(const Band &B, const double (&d)[SYS ? 15 : 10], const int iy, double b) {
    double A[5];
    coefficients(B, d, A);
    if constexpr (WALL) {
      if (iy == 1) {  // ghost then wall column
        const double e = A[0];
        for (int j = 1; j <= 4; j++) A[j] = A[j] - e * B.q->lo_ghost[j];
        const double f = A[1];
        for (int j = 2; j <= 4; j++) A[j] = A[j] - f * B.q->lo_wall[j];
        if (SYS == 0) b = b - A[1] * B.eta0 / B.bc0[1];
      } else if (iy == 2) {
        if (SYS == 0) b = b - A[0] * B.eta0 / B.bc0[1];
        const double e = A[0];
        for (int j = 1; j <= 3; j++) A[j] = A[j] - e * B.q->lo_wall[j + 1];
      }
      if (iy == B.ny - 1) {
        const double e = A[4];
        for (int j = 0; j <= 3; j++) A[j] = A[j] - e * B.q->hi_ghost[j];
        const double f = A[3];
        for (int j = 0; j <= 2; j++) A[j] = A[j] - f * B.q->hi_wall[j];
        if (SYS == 0) b = b - A[3] * B.etan / B.bcn[3];
        A[3] = 0.0;
        A[4] = 0.0;
      } else if (iy == B.ny - 2) {
        if (SYS == 0) b = b - A[4] * B.etan / B.bcn[3];
        const double e = A[4];
        for (int j = 1; j <= 3; j++) A[j] = A[j] - e * B.q->hi_wall[j - 1];
        A[4] = 0.0;
      }
    }
    step(A, b);
    return WALL ? make_double2(iy <= 2 ? 0.0 : A[0], iy == 1 ? 0.0 : A[1]) : make_double2(A[0], A[1]);
  }
};

// The rows ny-1 .. 1 of a bottom-up sweep: row(wall, iy, b) with the
// right-hand side b = load(iy) read N rows ahead into a register ring.
template <int N, class Load, class Row>
__device__ __forceinline__ void up_sweep(const int ny, Load load, Row row) {
  const double top[2] = {load(ny - 1), load(ny - 2)}, low[2] = {load(2), load(1)};
  double ring[N];  // ring[u] holds the right-hand side of row iy-u
#pragma unroll
  for (int u = 0; u < N; u++) ring[u] = load(max(ny - 3 - u, 1));
  const std::true_type wall{};
  const std::false_type inner{};
#pragma unroll 1
  for (int u = 0; u < 2; u++) row(wall, ny - 1 - u, u ? top[1] : top[0]);
  int iy = ny - 3;
  for (; iy - (N - 1) >= 3; iy -= N) {
#pragma unroll
    for (int u = 0; u < N; u++) {
      const int r = iy - u;
      const double b = ring[u];
      ring[u] = load(max(r - N, 1));
      row(inner, r, b);
    }
  }
#pragma unroll
  for (int u = 0; u < N; u++)
    if (iy - u >= 3) row(inner, iy - u, ring[u]);
#pragma unroll 1
  for (int u = 0; u < 2; u++) row(wall, 2 - u, u ? low[1] : low[0]);
}

// wall and ghost values from the three rows next to a wall (rows 1, 2, 3, or
// ny-3, ny-2, ny-1), linsolve_blocking.inc:50-61
__device__ __forceinline__ void wall_lo(const Band &B, const double *bot, double &w0, double &wm1) {
  const double s0 = B.bc0[2] * bot[0] + B.bc0[3] * bot[1] + B.bc0[4] * bot[2];
  w0 = (B.eta0 - s0) / B.bc0[1];
  const double s1 = B.bc0m1[1] * w0 + B.bc0m1[2] * bot[0] + B.bc0m1[3] * bot[1] + B.bc0m1[4] * bot[2];
  wm1 = -(s1 / B.bc0m1[0]);
}
__device__ __forceinline__ void wall_hi(const Band &B, double b3, double b2, double b1, double &wn, double &wp1) {
  const double s0 = B.bcn[0] * b3 + B.bcn[1] * b2 + B.bcn[2] * b1;
  wn = (B.etan - s0) / B.bcn[3];
  const double s1 = B.bcnp1[0] * b3 + B.bcnp1[1] * b2 + B.bcnp1[2] * b1 + B.bcnp1[3] * wn;
  wp1 = -(s1 / B.bcnp1[4]);
}

// ------------------------------------------------------------ k_solve_ve --
template <int SYS>
__device__ __forceinline__ void solve_column(const SolveArgs &a, const double *__restrict__ der) {
  // der is a separate restrict argument: the compiler then proves that the
  // kernel's stores never reach it and reads its wave-uniform rows through
  // the scalar cache, off the vector-memory counter that the sweeps' own
  // prefetches wait on.
  const Geom g = a.g;
  const int gid = xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
  // lane = 4*group + 2*sign + part; group (ix, |iz|) for iz >= 0, part 0 real,
  // 1 imaginary; the group after the last one solves ucor in pair slot npair
  const int grp = gid >> 2, sgn = (gid >> 1) & 1, part = gid & 1;
  const int ngrp = g.Nx * (g.nz + 1);
  if (grp > ngrp) return;
  const bool spare = grp == ngrp;
  const int ix = spare ? 0 : grp / (g.nz + 1), iza = spare ? 0 : grp % (g.nz + 1);
  if (sgn && (spare || iza == 0)) return;  // kz = 0 has no mirror
  const int iz = sgn ? -iza : iza;
  const int p = spare ? g.npair : ix * g.Nz + g.nz + iz;
  constexpr int sys = SYS;  // 0: eta (component 1), 1: v (component 2)
  const int ny = g.ny;
  const size_t gs = group_stride(ngrp);
  const double k2 = (g.alfa0 * ix) * (g.alfa0 * ix) + (g.beta0 * iz) * (g.beta0 * iz);
  const bool mean = !spare && ix == 0 && iz == 0;
  const size_t ps = g.ps, rs = 2 * ps;  // row stride in doubles
  double *col = reinterpret_cast<double *>(a.V + (size_t)sys * g.Ny * ps + p) + part;  // row iy at col[(iy+1)*rs]
  const double *rc = reinterpret_cast<const double *>(a.rhs + (size_t)sys * (ny - 1) * ps + p) + part;
  double2 *Lc = a.L + (size_t)sys * (ny - 1) * gs + grp;  // row iy at Lc[(iy-1)*gs]
  // wall value of eta: (Re u - Im w) + i (Im u + Re w) with u = u0/uN, w = 0
  // in the (0,0) mode, zero otherwise; v and dv/dy vanish at the walls.
  const double eta0 = (mean && sys == 0 && part == 0) ? a.u0 : 0.0;
  const double etan = (mean && sys == 0 && part == 0) ? a.uN : 0.0;
  const double bspare = (sys == 0 && part == 0) ? 1.0 : 0.0;  // ucor right-hand side

  // ---- bottom-up: rows, wall folding, factorisation, backward sweep
  const Band band(a, sys, k2, eta0, etan);
  UpState<SYS> st;
  auto up_row = [&](auto wall, const int iy, double b) {
    if (spare) b = bspare;
    double d[SYS ? 15 : 10];
#pragma unroll
    for (int j = 0; j < (SYS ? 15 : 10); j++) d[j] = der[(size_t)(iy - 1) * 20 + (j < 5 ? j : 5 + j)];
    const double2 L = st.template row<decltype(wall)::value>(band, d, iy, b);
    col[(size_t)(iy + 1) * rs] = st.x1;
    Lc[(size_t)(iy - 1) * gs] = L;
  };
  up_sweep<PF>(ny, [&](int r) { return rc[(size_t)(r - 1) * rs]; }, up_row);

  // ---- top-down: forward sweep, keep rows 1..3 and ny-3..ny-1
  double b1 = 0.0, b2 = 0.0, b3 = 0.0;
  double bot[3] = {0.0, 0.0, 0.0};
  auto down_row = [&](const int iy, const double x, const double2 L) {
    const double bi = x - (L.x * b2 + L.y * b1);
    col[(size_t)(iy + 1) * rs] = bi;
    if (iy <= 3) bot[iy - 1] = bi;
    b3 = b2;
    b2 = b1;
    b1 = bi;
  };
  {
    double xr[PF];
    double2 lr[PF];
#pragma unroll
    for (int u = 0; u < PF; u++) {
      const int r = min(1 + u, ny - 1);
      xr[u] = col[(size_t)(r + 1) * rs];
      lr[u] = Lc[(size_t)(r - 1) * gs];
    }
    int iy = 1;
    for (; iy + (PF - 1) <= ny - 1; iy += PF) {
#pragma unroll
      for (int u = 0; u < PF; u++) {
        const int r = iy + u;
        const double x = xr[u];
        const double2 L = lr[u];
        const int nr = min(r + PF, ny - 1);
        xr[u] = col[(size_t)(nr + 1) * rs];
        lr[u] = Lc[(size_t)(nr - 1) * gs];
        down_row(r, x, L);
      }
    }
#pragma unroll
    for (int u = 0; u < PF; u++)
      if (iy + u <= ny - 1) down_row(iy + u, xr[u], lr[u]);
  }
  // wall and ghost rows
  double w0, wm1, wn, wp1;
  wall_lo(band, bot, w0, wm1);
  wall_hi(band, b3, b2, b1, wn, wp1);
  col[rs] = w0;
  col[0] = wm1;
  col[(size_t)(ny + 1) * rs] = wn;
  col[(size_t)(ny + 2) * rs] = wp1;
}

__global__ __launch_bounds__(256, 5) void k_solve_ve(SolveArgs a, const double *__restrict__ der) {
  if (blockIdx.y)
    solve_column<1>(a, der);
  else
    solve_column<0>(a, der);
}

// One body for both systems, each pivot a division: slower by itself, but on grids that
// fill the memory system its waves stay closer together.  us per launch, this against
// k_solve_ve: 191x384x189 1004 and 1052 (4.5 waves per SIMD), 255x192x255 835 and 876 (8),
// 175x256x175 482 and 523 (3.8), 159x256x159 447 and 456 (3.1), but 143x256x143
// 389 and 350 (2.5), 127x384x127 539 and 486 (2): it is taken from three waves per
// SIMD on.  Its loops are its own: built from k_solve_ve's it took 1044.
__global__ __launch_bounds__(256) void k_solve_ve_wide(SolveArgs a, const double *__restrict__ der) {
  const Geom g = a.g;
  const int gid = xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
  const int grp = gid >> 2, sgn = (gid >> 1) & 1, part = gid & 1;
  const int ngrp = g.Nx * (g.nz + 1);
  if (grp > ngrp) return;
  const bool spare = grp == ngrp;
  const int ix = spare ? 0 : grp / (g.nz + 1), iza = spare ? 0 : grp % (g.nz + 1);
  if (sgn && (spare || iza == 0)) return;  // kz = 0 has no mirror
  const int iz = sgn ? -iza : iza;
  const int p = spare ? g.npair : ix * g.Nz + g.nz + iz;
  const int sys = blockIdx.y;  // 0: eta (component 1), 1: v (component 2)
  const int ny = g.ny;
  const size_t gs = group_stride(ngrp);
  const double k2 = (g.alfa0 * ix) * (g.alfa0 * ix) + (g.beta0 * iz) * (g.beta0 * iz);
  const bool mean = !spare && ix == 0 && iz == 0;
  const size_t ps = g.ps, rs = 2 * ps;  // row stride in doubles
  double *col = reinterpret_cast<double *>(a.V + (size_t)sys * g.Ny * ps + p) + part;  // row iy at col[(iy+1)*rs]
  const double *rc = reinterpret_cast<const double *>(a.rhs + (size_t)sys * (ny - 1) * ps + p) + part;
  double2 *Lc = a.L + (size_t)sys * (ny - 1) * gs + grp;  // row iy at Lc[(iy-1)*gs]
  const double *bc0 = a.bc[sys ? BC_V0 : BC_ETA0], *bc0m1 = a.bc[sys ? BC_V0M1 : BC_ETA0M1];
  const double *bcn = a.bc[sys ? BC_VN : BC_ETAN], *bcnp1 = a.bc[sys ? BC_VNP1 : BC_ETANP1];
  const double eta0 = (mean && sys == 0 && part == 0) ? a.u0 : 0.0;
  const double etan = (mean && sys == 0 && part == 0) ? a.uN : 0.0;
  const double bspare = (sys == 0 && part == 0) ? 1.0 : 0.0;  // ucor right-hand side

  // ---- bottom-up: rows, wall folding, factorisation, backward sweep
  double l1m2 = 0.0, l1m1 = 0.0, l2m2 = 0.0, l2m1 = 0.0;  // lower factors of rows iy+1, iy+2
  double x1 = 0.0, x2 = 0.0;
  auto up_row = [&](const int iy, double b) {
    if (spare) b = bspare;
    const double *d = der + (size_t)(iy - 1) * 20;
    double A[5];
#pragma unroll
    for (int j = 0; j < 5; j++) {
      const double d0 = d[j], d2 = d[10 + j], d4 = d[15 + j];
      if (sys) {
        const double os = a.ni * (d4 - 2.0 * k2 * d2 + k2 * k2 * d0);
        A[j] = a.lambda * (d2 - k2 * d0) - os;
      } else {
        const double sq = a.ni * (d2 - k2 * d0);
        A[j] = a.lambda * d0 - sq;
      }
    }
    if (iy == 1) {  // applybc_0 row 1: ghost then wall column
      const double e = A[0];
      for (int j = 1; j <= 4; j++) A[j] = A[j] - e * bc0m1[j] / bc0m1[0];
      const double f = A[1];
      for (int j = 2; j <= 4; j++) A[j] = A[j] - f * bc0[j] / bc0[1];
      if (sys == 0) b = b - A[1] * eta0 / bc0[1];
    } else if (iy == 2) {
      if (sys == 0) b = b - A[0] * eta0 / bc0[1];
      const double e = A[0];
      for (int j = 1; j <= 3; j++) A[j] = A[j] - e * bc0[j + 1] / bc0[1];
    }
    if (iy == ny - 1) {  // applybc_n row ny-1
      const double e = A[4];
      for (int j = 0; j <= 3; j++) A[j] = A[j] - e * bcnp1[j] / bcnp1[4];
      const double f = A[3];
      for (int j = 0; j <= 2; j++) A[j] = A[j] - f * bcn[j] / bcn[3];
      if (sys == 0) b = b - A[3] * etan / bcn[3];
      A[3] = 0.0;
      A[4] = 0.0;
    } else if (iy == ny - 2) {
      if (sys == 0) b = b - A[4] * etan / bcn[3];
      const double e = A[4];
      for (int j = 1; j <= 3; j++) A[j] = A[j] - e * bcn[j - 1] / bcn[3];
      A[4] = 0.0;
    }
    // factorise row iy against the already factorised rows iy+1, iy+2
    const double p2 = A[4];
    A[3] = A[3] - p2 * l2m1;
    A[2] = A[2] - p2 * l2m2;
    const double p1 = A[3];
    A[2] = A[2] - p1 * l1m1;
    A[1] = A[1] - p1 * l1m2;
    const double r = 1.0 / A[2];
    A[0] = A[0] * r;
    A[1] = A[1] * r;
    // backward sweep
    const double xi = (b - (p1 * x1 + p2 * x2)) * r;
    col[(size_t)(iy + 1) * rs] = xi;
    Lc[(size_t)(iy - 1) * gs] = make_double2(iy <= 2 ? 0.0 : A[0], iy == 1 ? 0.0 : A[1]);
    l2m2 = l1m2;
    l2m1 = l1m1;
    l1m2 = A[0];
    l1m1 = A[1];
    x2 = x1;
    x1 = xi;
  };
  {
    double ring[PF];  // ring[u] holds the right-hand side of row iy-u
#pragma unroll
    for (int u = 0; u < PF; u++) ring[u] = rc[(size_t)max(ny - 2 - u, 0) * rs];
    int iy = ny - 1;
    for (; iy - (PF - 1) >= 1; iy -= PF) {
#pragma unroll
      for (int u = 0; u < PF; u++) {
        const int r = iy - u;
        const double b = ring[u];
        ring[u] = rc[(size_t)max(r - PF - 1, 0) * rs];
        up_row(r, b);
      }
    }
#pragma unroll
    for (int u = 0; u < PF; u++)
      if (iy - u >= 1) up_row(iy - u, ring[u]);
  }

  // ---- top-down: forward sweep, keep rows 1..3 and ny-3..ny-1
  double b1 = 0.0, b2 = 0.0, b3 = 0.0;
  double bot[3] = {0.0, 0.0, 0.0};
  auto down_row = [&](const int iy, const double x, const double2 L) {
    const double bi = x - (L.x * b2 + L.y * b1);
    col[(size_t)(iy + 1) * rs] = bi;
    if (iy <= 3) bot[iy - 1] = bi;
    b3 = b2;
    b2 = b1;
    b1 = bi;
  };
  {
    double xr[PF];
    double2 lr[PF];
#pragma unroll
    for (int u = 0; u < PF; u++) {
      const int r = min(1 + u, ny - 1);
      xr[u] = col[(size_t)(r + 1) * rs];
      lr[u] = Lc[(size_t)(r - 1) * gs];
    }
    int iy = 1;
    for (; iy + (PF - 1) <= ny - 1; iy += PF) {
#pragma unroll
      for (int u = 0; u < PF; u++) {
        const int r = iy + u;
        const double x = xr[u];
        const double2 L = lr[u];
        const int nr = min(r + PF, ny - 1);
        xr[u] = col[(size_t)(nr + 1) * rs];
        lr[u] = Lc[(size_t)(nr - 1) * gs];
        down_row(r, x, L);
      }
    }
#pragma unroll
    for (int u = 0; u < PF; u++)
      if (iy + u <= ny - 1) down_row(iy + u, xr[u], lr[u]);
  }
  // wall and ghost rows
  {
    const double s0 = bc0[2] * bot[0] + bc0[3] * bot[1] + bc0[4] * bot[2];
    const double w0 = (eta0 - s0) / bc0[1];
    const double s1 = bc0m1[1] * w0 + bc0m1[2] * bot[0] + bc0m1[3] * bot[1] + bc0m1[4] * bot[2];
    const double wm1 = sys ? (0.0 - s1) / bc0m1[0] : -(s1 / bc0m1[0]);
    col[rs] = w0;
    col[0] = wm1;
  }
  {
    const double s0 = bcn[0] * b3 + bcn[1] * b2 + bcn[2] * b1;  // rows ny-3, ny-2, ny-1
    const double wn = (etan - s0) / bcn[3];
    const double s1 = bcnp1[0] * b3 + bcnp1[1] * b2 + bcnp1[2] * b1 + bcnp1[3] * wn;
    const double wp1 = sys ? (0.0 - s1) / bcnp1[4] : -(s1 / bcnp1[4]);
    col[(size_t)(ny + 1) * rs] = wn;
    col[(size_t)(ny + 2) * rs] = wp1;
  }
}

// ---------------------------------------------------------------- k_mean --
// yintegr (dnsdata.f90:312-324): the three-point rule on the odd rows; f and y
// are indexed by row + 1.  Term t covers rows 2t+1 .. 2t+3.
__device__ __forceinline__ double yintegr_term(const double *y, const double *f, int iy) {
  const double yp1 = y[iy + 2] - y[iy + 1], ym1 = y[iy] - y[iy + 1];
  const double a1 = -(1.0 / 3.0 * ym1) + 1.0 / 6.0 * yp1 + 1.0 / 6.0 * yp1 * yp1 / ym1;
  const double a3 = +(1.0 / 3.0 * yp1) - 1.0 / 6.0 * ym1 - 1.0 / 6.0 * ym1 * ym1 / yp1;
  const double a2 = yp1 - ym1 - a1 - a3;
  return a1 * f[iy] + a2 * f[iy + 1] + a3 * f[iy + 2];
}

// Sums yintegr of nf columns (stride Ny in LDS) with the block; red holds
// nf*256 doubles.  Every thread of the block calls it.
template <int NF>
__device__ void yintegr_block(const double *y, const double *f, int Ny, int ny, double *red, double *out) {
  double s[NF];
#pragma unroll
  for (int k = 0; k < NF; k++) s[k] = 0.0;
  for (int iy = 1 + 2 * (int)threadIdx.x; iy <= ny - 1; iy += 2 * (int)blockDim.x)
#pragma unroll
    for (int k = 0; k < NF; k++) s[k] += yintegr_term(y, f + k * Ny, iy);
#pragma unroll
  for (int k = 0; k < NF; k++) red[k * 256 + threadIdx.x] = s[k];
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h)
#pragma unroll
      for (int k = 0; k < NF; k++) red[k * 256 + threadIdx.x] += red[k * 256 + threadIdx.x + h];
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < NF; k++) out[k] = red[k * 256];
}

__global__ __launch_bounds__(256) void k_mean(MeanArgs a) {
  extern __shared__ double sm[];
  const Geom g = a.g;
  const int Ny = g.Ny, ny = g.ny;
  const size_t ps = g.ps, pstride = (size_t)Ny * ps;
  const int p0 = g.nz;  // pair (ix=0, iz=0)
  double *ur = sm, *wr = sm + Ny, *uc = sm + 2 * Ny, *yy = sm + 3 * Ny, *red = sm + 4 * Ny;
  __shared__ double cv[4];  // flag x, flag z, corrpx, corrpz
  for (int i = threadIdx.x; i < Ny; i += blockDim.x) {
    const cx<double> e = a.V[(size_t)i * ps + p0];  // eta slot: Re u + i Re w
    ur[i] = e.x;
    wr[i] = e.y;
    uc[i] = a.V[(size_t)i * ps + g.npair].x;  // ucor from the spare slot
    yy[i] = a.y[i];
  }
  __syncthreads();
  double fr[3];
  yintegr_block<3>(yy, sm, Ny, ny, red, fr);
  if (threadIdx.x == 0) {
    DevScalars *sc = a.sc;
    sc->fr[0] = fr[0];
    sc->fr[1] = fr[1];
    sc->fr[2] = fr[2];
    cv[0] = 0.0;
    cv[1] = 0.0;
    if (fabs(a.meanflowx) > 1.0e-7 && !a.cpi) {
      sc->corrpx = (a.meanflowx - fr[0]) / fr[2];
      cv[0] = 1.0;
    }
    if (fabs(a.meanflowz) > 1.0e-7 && !a.cpi) {
      sc->corrpz = (a.meanflowz - fr[1]) / fr[2];
      cv[1] = 1.0;
    }
    cv[2] = sc->corrpx;
    cv[3] = sc->corrpz;
    if (a.cpi) {
      if (a.cpi_type == 0)
        sc->meanpx = (1 - a.gamma) * 6 * a.ni / fr[0];
      else
        sc->meanpx = (1.5 / a.gamma) * fr[0] * a.ni;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < Ny; i += blockDim.x) {
    double u = ur[i], w = wr[i];
    if (cv[0] != 0.0) u = u + cv[2] * uc[i];
    if (cv[1] != 0.0) w = w + cv[3] * uc[i];
    a.V[(size_t)i * ps + p0] = cx<double>{u, 0.0};
    a.V[2 * pstride + (size_t)i * ps + p0] = cx<double>{w, 0.0};
  }
}

// ------------------------------------------------------------------ dv/dy --
__device__ __forceinline__ double dot5(const double *w, const double *v) {
  double s = w[0] * v[0];
#pragma unroll
  for (int j = 1; j < 5; j++) s = s + w[j] * v[j];
  return s;
}

// row iy of the bottom-up D0 sweep: D1 v (w[j] = v(iy-2+j)) with the wall and
// ghost derivatives' columns taken to the right, then the substitution; d0,
// d1 the row's stencils, D its factors
__device__ __forceinline__ double dv_up(const double *d0, const double *d1, const double *D, const int iy, const int ny,
                                        const double *w, double f10, double f1m1, double f1n, double f1np1, double x1,
                                        double x2) {
  double f = dot5(d1, w);
  if (iy == ny - 1) f = f - (d0[3] * f1n + d0[4] * f1np1);
  if (iy == ny - 2) f = f - d0[4] * f1n;
  if (iy == 2) f = f - d0[0] * f10;
  if (iy == 1) f = f - (d0[1] * f10 + d0[0] * f1m1);
  return (f - (D[3] * x1 + D[4] * x2)) * D[2];
}

// ------------------------------------------------------------------ k_uw --
// Blocks of two waves: the kernel has few waves (one lane per pair and part)
// and each runs a long sequential sweep, so smaller blocks spread them more
// evenly over the CUs (5% faster than 256-thread blocks at 191x384x189).
constexpr int UW_BLOCK = 128;
__global__ __launch_bounds__(UW_BLOCK) void k_uw(UwArgs a, const double *__restrict__ der, const double *__restrict__ d0fac) {
  const Geom g = a.g;
  const int gid = blockIdx.x * UW_BLOCK + threadIdx.x;
  const int p = gid >> 1, part = gid & 1;  // part 0 real, 1 imaginary
  if (p >= g.npair) return;
  const int ix = p / g.Nz, iz = p % g.Nz - g.nz;
  if (ix == 0 && iz == 0) return;  // both lanes of the (0,0) pair leave together
  const int ny = g.ny;
  const double al = g.alfa0 * ix, be = g.beta0 * iz;
  const double k2 = (g.alfa0 * ix) * (g.alfa0 * ix) + (g.beta0 * iz) * (g.beta0 * iz);
  const size_t ps = g.ps, rs = 2 * ps, pstride = (size_t)g.Ny * ps;
  double *c1 = reinterpret_cast<double *>(a.V + p) + part;
  double *c2 = reinterpret_cast<double *>(a.V + pstride + p) + part;
  double *c3 = reinterpret_cast<double *>(a.V + 2 * pstride + p) + part;
#define ROW(c, iy) (c)[(size_t)((iy) + 1) * rs]
  // one-sided wall and ghost derivatives of this part of v
  double vb[5], vt[5];
#pragma unroll
  for (int j = 0; j < 5; j++) {
    vb[j] = ROW(c2, -1 + j);
    vt[j] = ROW(c2, ny - 3 + j);
  }
  const double f10 = dot5(a.bnd[B_D140], vb), f1m1 = dot5(a.bnd[B_D14M1], vb);
  const double f1n = dot5(a.bnd[B_D14N], vt), f1np1 = dot5(a.bnd[B_D14NP1], vt);

  // bottom-up: interior D1 v with boundary fix-ups and the D0 backward sweep;
  // window w[j] = v(iy-2+j)
  double w[5];
#pragma unroll
  for (int j = 0; j < 5; j++) w[j] = vt[j];
  double x1 = f1n, x2 = f1np1;
  auto up_row = [&](const int iy, const double vnext) {  // vnext = v(iy-3)
    const double *d = der + (size_t)(iy - 1) * 20;
    const double xi = dv_up(d, d + 5, d0fac + (size_t)(iy - 1) * 5, iy, ny, w, f10, f1m1, f1n, f1np1, x1, x2);
    ROW(c3, iy) = xi;
    x2 = x1;
    x1 = xi;
#pragma unroll
    for (int j = 4; j > 0; j--) w[j] = w[j - 1];
    w[0] = vnext;
  };
  {
    double ring[PF];  // ring[u] holds v(iy-u-3)
#pragma unroll
    for (int u = 0; u < PF; u++) ring[u] = ROW(c2, max(ny - 4 - u, -1));
    int iy = ny - 1;
    for (; iy - (PF - 1) >= 1; iy -= PF) {
#pragma unroll
      for (int u = 0; u < PF; u++) {
        const int r = iy - u;
        const double v = ring[u];
        ring[u] = ROW(c2, max(r - 3 - PF, -1));
        up_row(r, v);
      }
    }
#pragma unroll
    for (int u = 0; u < PF; u++)
      if (iy - u >= 1) up_row(iy - u, ring[u]);
  }

  // top-down: D0 forward sweep, then u and w on every row; the other part of
  // v' and eta comes from the neighbouring lane
  double b1 = f10, b2 = f1m1;
  auto down_row = [&](const int iy, const double x, const double eta) {
    double vp;
    if (iy == -1)
      vp = f1m1;
    else if (iy == 0)
      vp = f10;
    else if (iy <= ny - 1) {
      const double *D = d0fac + (size_t)(iy - 1) * 5;
      vp = x - (D[0] * b2 + D[1] * b1);
      b2 = b1;
      b1 = vp;
    } else
      vp = iy == ny ? f1n : f1np1;
    const double vo = __shfl_xor(vp, 1, 64), eo = __shfl_xor(eta, 1, 64);
    // u = (i al v' - i be eta)/k2, w = (i be v' + i al eta)/k2, i*a*X = (-a Xi, a Xr)
    double uu, ww;
    if (part == 0) {
      uu = (-(al * vo)) - (-(be * eo));
      ww = (-(be * vo)) + (-(al * eo));
    } else {
      uu = (al * vo) - (be * eo);
      ww = (be * vo) + (al * eo);
    }
    ROW(c1, iy) = uu / k2;
    ROW(c3, iy) = ww / k2;
  };
  {
    double xr[PF], er[PF];  // D1 v / D0 backward result and eta of row iy+u
#pragma unroll
    for (int u = 0; u < PF; u++) {
      xr[u] = ROW(c3, -1 + u);
      er[u] = ROW(c1, -1 + u);
    }
    int iy = -1;
    for (; iy + (PF - 1) <= ny + 1; iy += PF) {
#pragma unroll
      for (int u = 0; u < PF; u++) {
        const int r = iy + u;
        const double x = xr[u], e = er[u];
        const int nr = min(r + PF, ny + 1);
        xr[u] = ROW(c3, nr);
        er[u] = ROW(c1, nr);
        down_row(r, x, e);
      }
    }
#pragma unroll
    for (int u = 0; u < PF; u++)
      if (iy + u <= ny + 1) down_row(iy + u, xr[u], er[u]);
  }
#undef ROW
}

// ---------------------------------------------------------- k_solve_lds --
// The whole of linsolve but the (0,0) mode's flow-rate correction in one
// kernel, for grids whose columns fit in LDS: a block of four waves holds 16
// (kx, |kz|) groups of both systems as X[sys][row][64] in LDS, waves 0 and 1
// eta, 2 and 3 v, 8 groups each.  What bounds it is the length of the dependent
// chain of rows, so every column is swept from both walls at once: lanes 0..31
// of a wave eliminate from the upper wall down to row m+1, lanes 32..63 from
// the lower wall up to row m, m = (ny-1)/2, in the mirrored frame k = 1, 2, ..
// from their own wall with mirrored stencils, so that both halves run the same
// code.  The two innermost rows of each half close a 2x2 system, and both halves
// substitute outwards.  The D0 solve of dv/dy (waves 2 and 3, in place) goes
// the same way, with its factors from the set-up.  The block then writes u, v
// and w: nothing of the intermediate columns goes through memory (nor do the
// lower factors when they fit beside the columns, LLDS).  Against k_solve_ve
// and k_uw (FP64, us per substep): 15x32x15 14.5 for 46.8, 31x64x31 23.9 for 89,
// 63x96x47 35 for 146, 95x128x95 117 for 223, 191x128x189 377 for 497; one
// sweep per column in the same LDS layout took 34.7 at 31x64x31 and 190 at
// 95x128x95.
//
// The rows' stencils come from a staged table one row ahead (from the scalar
// cache every row waits for them), the two systems have their own code, and no
// lane is masked: the mirror lanes of kz = 0 and those past the last group
// repeat another lane's column and store the same values.
constexpr int SPF = 8;

// A lane's half of a column: offsets of row k = 0 and from row k to k + 1.
struct Half {
  int up;  // 1: the lower wall's half (rows k), 0: the upper wall's (rows ny - k)
  int x0, xs, t0, ts, l0, ls;
  __device__ __forceinline__ Half(int up, int ny) : up(up) {
    x0 = (up ? 1 : ny + 1) * 64;
    xs = up ? 64 : -64;
    t0 = (up ? -1 : ny - 1) * SROW;
    ts = up ? SROW : -SROW;
    l0 = up ? -1 : ny - 1;
    ls = up ? 1 : -1;
  }
};

// The innermost unknowns of the other half, b1 next to the meeting point and b2
// behind it, from the last two rows of each half: x + p1 b1 + p2 b2 = a and
// x' + q1 x + q2 b1 = c with x, x' this half's innermost unknowns.
__device__ __forceinline__ void meet(double a, double p1, double p2, double c, double q1, double q2, double &b1, double &b2) {
  auto other = [](double v) { return __shfl_xor(v, 32, 64); };
  const double A = other(a), P1 = other(p1), P2 = other(p2), C = other(c), Q1 = other(q1), Q2 = other(q2);
  const double m11 = 1.0 - p2 * Q2, m12 = p1 - p2 * Q1, r1 = a - p2 * C;
  const double m21 = P1 - P2 * q1, m22 = 1.0 - P2 * q2, r2 = A - P2 * c;
  const double det = m11 * m22 - m12 * m21;
  const double x = (r1 * m22 - m12 * r2) / det;
  b1 = (m11 * r2 - m21 * r1) / det;
  b2 = C - Q1 * b1 - Q2 * x;
}

// Rows k = 1 .. m of both halves, then row m + 1 of the upper one when ny - 1 is
// odd: row(wall, k, b) with b = load(k) read N rows ahead.
template <int N, class Load, class Row>
__device__ __forceinline__ void inward(const int m, const bool more, Load load, Row row) {
  const double b1 = load(1), b2 = load(2), last = more ? load(m + 1) : 0.0;
  double ring[N];
#pragma unroll
  for (int u = 0; u < N; u++) ring[u] = load(min(3 + u, m));
  const std::true_type wall{};
  const std::false_type inner{};
#pragma unroll 1
  for (int k = 1; k <= 2; k++) row(wall, k, k == 1 ? b1 : b2);
  int k = 3;
  for (; k + (N - 1) <= m; k += N) {
#pragma unroll
    for (int u = 0; u < N; u++) {
      const double b = ring[u];
      ring[u] = load(min(k + u + N, m));
      row(inner, k + u, b);
    }
  }
#pragma unroll
  for (int u = 0; u < N; u++)
    if (k + u <= m) row(inner, k + u, ring[u]);
  if (more) row(inner, m + 1, last);
}

template <int SYS, bool LLDS>
__device__ __forceinline__ void lds_sweeps(const SolveArgs &a, const Band &band, const Half h, const double *T, double *x,
                                           double2 *Ls, double2 *Lg, size_t gs, const double *rc, double *gcol, size_t rs,
                                           bool spare, double bspare) {
  constexpr int ND = SYS ? 15 : 10;
  const int ny = band.ny, m = (ny - 1) / 2;
  const bool more = ((ny - 1) & 1) && !h.up;
  // the wall rows in the mirrored frame
  const double wv = h.up ? band.eta0 : band.etan;
  double gh[4], wl[3], w3[3], g4[4];
  const double *bw = h.up ? band.bc0 : band.bcn, *bg = h.up ? band.bc0m1 : band.bcnp1;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    gh[j] = h.up ? band.q->lo_ghost[4 - j] : band.q->hi_ghost[j];
    g4[j] = bg[h.up ? 4 - j : j];
    if (j < 3) {
      wl[j] = h.up ? band.q->lo_wall[4 - j] : band.q->hi_wall[j];
      w3[j] = bw[h.up ? 4 - j : j];
    }
  }
  const double wd = bw[h.up ? 1 : 3], gd = bg[h.up ? 0 : 4];
  UpState<SYS> st;
  {
    double dn[ND];
#pragma unroll
    for (int j = 0; j < ND; j++) dn[j] = T[h.t0 + h.ts + j];
    auto row = [&](auto wall, const int k, double b) {
      if (spare) b = bspare;
      double d[ND], A[5];
      const double *Tn = T + h.t0 + min(k + 1, m + 1) * h.ts;
#pragma unroll
      for (int j = 0; j < ND; j++) {
        d[j] = dn[j];
        dn[j] = Tn[j];
      }
      st.coefficients(band, d, A);
      if constexpr (decltype(wall)::value) {
        if (k == 1) {  // ghost then wall column
          const double e = A[4];
          for (int j = 0; j < 4; j++) A[j] -= e * gh[j];
          const double f = A[3];
          for (int j = 0; j < 3; j++) A[j] -= f * wl[j];
          if (SYS == 0) b -= A[3] * wv / wd;
          A[3] = 0.0;
        } else {
          const double e = A[4];
          if (SYS == 0) b -= e * wv / wd;
          for (int j = 1; j < 4; j++) A[j] -= e * wl[j - 1];
        }
        A[4] = 0.0;
      }
      st.step(A, b);
      x[h.x0 + k * h.xs] = st.x1;
      // the group's four lanes have the same factors
      if constexpr (LLDS)
        Ls[(h.l0 + k * h.ls) * 16] = make_double2(A[0], A[1]);
      else
        Lg[(size_t)(h.l0 + k * h.ls) * gs] = make_double2(A[0], A[1]);
    };
    inward<SPF>(m, more, [&](int k) { return rc[(size_t)(h.l0 + k * h.ls) * rs]; }, row);
  }
  // ---- outwards; v goes to memory
  double b1, b2;
  meet(st.x1, st.l1m1, st.l1m2, st.x2, st.l2m1, st.l2m2, b1, b2);
  auto out = [&](const int k, const double xv, const double2 L) {
    const double bi = xv - (L.x * b2 + L.y * b1);
    x[h.x0 + k * h.xs] = bi;
    if constexpr (SYS) gcol[(size_t)(h.l0 + k * h.ls + 2) * rs] = bi;
    b2 = b1;
    b1 = bi;
  };
  if (more) out(m + 1, st.x1, make_double2(st.l1m2, st.l1m1));
  constexpr int DP = LLDS ? 4 : SPF;
  double xr[DP];
  double2 lr[DP];
  auto fetch = [&](int k, int u) {
    xr[u] = x[h.x0 + k * h.xs];
    if constexpr (LLDS)
      lr[u] = Ls[(h.l0 + k * h.ls) * 16];
    else
      lr[u] = Lg[(size_t)(h.l0 + k * h.ls) * gs];
  };
#pragma unroll
  for (int u = 0; u < DP; u++) fetch(max(m - u, 1), u);
  int k = m;
  for (; k - (DP - 1) >= 1; k -= DP) {
#pragma unroll
    for (int u = 0; u < DP; u++) {
      const double xv = xr[u];
      const double2 L = lr[u];
      fetch(max(k - u - DP, 1), u);
      out(k - u, xv, L);
    }
  }
#pragma unroll
  for (int u = 0; u < DP; u++)
    if (k - u >= 1) out(k - u, xr[u], lr[u]);
  // wall and ghost rows (k = 0 and -1) from the rows 3, 2, 1
  const double c3 = x[h.x0 + 3 * h.xs], c2 = x[h.x0 + 2 * h.xs], c1 = x[h.x0 + h.xs];
  const double w = (wv - (w3[0] * c3 + w3[1] * c2 + w3[2] * c1)) / wd;
  const double g = -(g4[0] * c3 + g4[1] * c2 + g4[2] * c1 + g4[3] * w) / gd;
  x[h.x0] = w;
  x[h.x0 - h.xs] = g;
  if constexpr (SYS) {
    gcol[(size_t)(h.l0 + 2) * rs] = w;
    gcol[(size_t)(h.l0 - h.ls + 2) * rs] = g;
  }
}

// Orders a wave's LDS accesses where its lanes exchange data.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// dv/dy of the v columns x, in place.  The stencils of the innermost rows reach
// three rows of the other half, which its lanes of the same wave overwrite: they
// are taken between two fences, before either half starts.
__device__ __forceinline__ void lds_dv(const UwArgs &uw, const Half h, const double *T, double *x, const int ny) {
  const int m = (ny - 1) / 2;
  const bool more = ((ny - 1) & 1) && !h.up;
  wave_sync();
  double vo[3];  // v of the rows m + 1 .. m + 3
#pragma unroll
  for (int j = 0; j < 3; j++) vo[j] = x[h.x0 + (m + 1 + j) * h.xs];
  wave_sync();
  // one-sided derivatives at the wall (fw) and the ghost row (fg): the window
  // w[j] = v of row k + 2 - j in the mirrored frame, here at k = 1
  double w[5], fw = 0.0, fg = 0.0;
#pragma unroll
  for (int j = 0; j < 5; j++) {
    w[j] = x[h.x0 + (3 - j) * h.xs];
    fw += w[j] * (h.up ? uw.bnd[B_D140][4 - j] : uw.bnd[B_D14N][j]);
    fg += w[j] * (h.up ? uw.bnd[B_D14M1][4 - j] : uw.bnd[B_D14NP1][j]);
  }
  constexpr int U = 4;
  double x1 = 0.0, x2 = 0.0, vr[U], dr[U][8];  // v of row k + 3, d1 and the factors D[2..4] of the rows ahead
  auto fetch = [&](int k, int u) {
    vr[u] = x[h.x0 + min(k + 3, m) * h.xs];
    const double *t = T + h.t0 + min(k, m + 1) * h.ts;
#pragma unroll
    for (int j = 0; j < 5; j++) dr[u][j] = t[15 + j];
#pragma unroll
    for (int j = 0; j < 3; j++) dr[u][5 + j] = t[22 + j];
  };
  auto in = [&](auto inner, int k, int u, double g) {
    double vnext = vr[u];
    if constexpr (decltype(inner)::value)
      if (k + 3 > m) vnext = k + 2 == m ? vo[0] : (k + 1 == m ? vo[1] : vo[2]);
    double d[8];
#pragma unroll
    for (int j = 0; j < 8; j++) d[j] = dr[u][j];
    fetch(k + U, u);
    const double f = dot5(d, w) - g;
    const double xi = (f - (d[6] * x1 + d[7] * x2)) * d[5];
    x[h.x0 + k * h.xs] = xi;
    x2 = x1;
    x1 = xi;
#pragma unroll
    for (int j = 4; j > 0; j--) w[j] = w[j - 1];
    w[0] = vnext;
  };
#pragma unroll
  for (int u = 0; u < U; u++) fetch(1 + u, u);
  // the wall and ghost derivatives' columns of the rows 1 and 2
  const double *t1 = T + h.t0 + h.ts;
  const double g1 = t1[3] * fw + t1[4] * fg, g2 = t1[h.ts + 4] * fw;
  int k = 1;
  for (; k + (U - 1) <= m - 3; k += U) {  // rows whose stencils stay in this half
#pragma unroll
    for (int u = 0; u < U; u++) in(std::false_type{}, k + u, u, u == 0 ? (k == 1 ? g1 : 0.0) : (u == 1 && k == 1 ? g2 : 0.0));
  }
#pragma unroll 1
  for (; k <= m; k += U) {
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k + u <= m) in(std::true_type{}, k + u, u, k + u == 1 ? g1 : (k + u == 2 ? g2 : 0.0));
  }
  if (more) {
    double d[5], D[3];
    const double *t = T + h.t0 + (m + 1) * h.ts;
#pragma unroll
    for (int j = 0; j < 5; j++) d[j] = t[15 + j];
#pragma unroll
    for (int j = 0; j < 3; j++) D[j] = t[22 + j];
    const double xi = (dot5(d, w) - (D[1] * x1 + D[2] * x2)) * D[0];
    x2 = x1;
    x1 = xi;
  }
  const double *tl = T + h.t0 + (more ? m + 1 : m) * h.ts;
  double b1, b2;
  meet(x1, tl[21], tl[20], x2, tl[21 - h.ts], tl[20 - h.ts], b1, b2);
  if (more) {
    const double vp = x1 - (tl[20] * b2 + tl[21] * b1);
    x[h.x0 + (m + 1) * h.xs] = vp;
    b2 = b1;
    b1 = vp;
  }
  double xr[U], Dr[U][2];
  auto fetch2 = [&](int k, int u) {
    xr[u] = x[h.x0 + k * h.xs];
    const double *t = T + h.t0 + k * h.ts;
    Dr[u][0] = t[20];
    Dr[u][1] = t[21];
  };
  auto out = [&](int k, int u) {
    const double vp = xr[u] - (Dr[u][0] * b2 + Dr[u][1] * b1);
    fetch2(max(k - U, 1), u);
    x[h.x0 + k * h.xs] = vp;
    b2 = b1;
    b1 = vp;
  };
#pragma unroll
  for (int u = 0; u < U; u++) fetch2(max(m - u, 1), u);
  k = m;
  for (; k - (U - 1) >= 1; k -= U) {
#pragma unroll
    for (int u = 0; u < U; u++) out(k - u, u);
  }
#pragma unroll
  for (int u = 0; u < U; u++)
    if (k - u >= 1) out(k - u, u);
  x[h.x0] = fw;
  x[h.x0 - h.xs] = fg;
}

template <bool LLDS>
__global__ __launch_bounds__(256) void k_solve_lds(SolveArgs a, UwArgs uw, const double *__restrict__ tab) {
  extern __shared__ __align__(16) double smem[];
  const Geom g = a.g;
  const int ny = g.ny, ngrp = g.Nx * (g.nz + 1);
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  if (blk * 16 > ngrp) return;  // the whole block: padding of the grid
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), sys = wave >> 1, l = threadIdx.x & 63;
  const int lg = 8 * (wave & 1) + ((l >> 2) & 7);  // the block's group; lane = 32*half + 4*(group % 8) + 2*sign + part
  const int grp = min(blk * 16 + lg, ngrp), sgn = (l >> 1) & 1, part = l & 1;
  const bool spare = grp == ngrp;
  const int ix = spare ? 0 : grp / (g.nz + 1), iza = spare ? 0 : grp % (g.nz + 1);
  const int iz = sgn ? -iza : iza;
  const int p = spare ? g.npair : ix * g.Nz + g.nz + iz;
  const size_t gs = group_stride(ngrp);
  const double k2 = (g.alfa0 * ix) * (g.alfa0 * ix) + (g.beta0 * iz) * (g.beta0 * iz);
  const bool mean = !spare && ix == 0 && iz == 0;
  const size_t ps = g.ps, rs = 2 * ps;
  const int column = 32 * (wave & 1) + (l & 31);
  const Half h(l >> 5, ny);
  double *X0 = smem, *X1 = X0 + (size_t)(ny + 3) * 64;  // eta and v columns, row iy at [(iy+1)*64 + column]
  double *T = X1 + (size_t)(ny + 3) * 64;               // the table
  double2 *Ls = reinterpret_cast<double2 *>(T + (size_t)(ny - 1) * SROW) + (size_t)sys * (ny - 1) * 16 + lg;
  double2 *Lg = a.L + (size_t)sys * (ny - 1) * gs + grp;
  const double *rc = reinterpret_cast<const double *>(a.rhs + (size_t)sys * (ny - 1) * ps + p) + part;
  double *gcol = reinterpret_cast<double *>(a.V + (size_t)sys * g.Ny * ps + p) + part;  // row iy at gcol[(iy+1)*rs]
  const double eta0 = (mean && sys == 0 && part == 0) ? a.u0 : 0.0;
  const double etan = (mean && sys == 0 && part == 0) ? a.uN : 0.0;
  const double bspare = (sys == 0 && part == 0) ? 1.0 : 0.0;
  const Band band(a, sys, k2, eta0, etan);
  {
    const double2 *t2 = reinterpret_cast<const double2 *>(tab);
    double2 *T2 = reinterpret_cast<double2 *>(T);
#pragma unroll 4
    for (int i = threadIdx.x; i < (ny - 1) * (SROW / 2); i += 256) T2[i] = t2[i];
  }
  __syncthreads();
  if (sys) {
    lds_sweeps<1, LLDS>(a, band, h, T, X1 + column, Ls, Lg, gs, rc, gcol, rs, spare, bspare);
    lds_dv(uw, h, T, X1 + column, ny);
  } else {
    lds_sweeps<0, LLDS>(a, band, h, T, X0 + column, Ls, Lg, gs, rc, gcol, rs, spare, bspare);
    // eta itself is wanted only of the (0,0) mode and of ucor (k_mean)
    if (mean || spare)
      for (int r = h.up; r < ny + 3; r += 2) gcol[(size_t)r * rs] = X0[r * 64 + column];
  }
  __syncthreads();

  // ---- u (waves 0 and 1) and w (2 and 3) from the other part of v' and eta;
  // the half waves take alternate rows
  if (mean || spare) return;
  const double al = g.alfa0 * ix, be = g.beta0 * iz, rk = 1.0 / k2;
  // part 0: u = be eta - al v', w = -(be v' + al eta); part 1: the negatives
  const double *vo = X1 + (column ^ 1), *eo = X0 + (column ^ 1);
  const double cv = sys ? (part ? be : -be) : (part ? al : -al), ce = sys ? (part ? al : -al) : (part ? -be : be);
  double *out = reinterpret_cast<double *>(a.V + (size_t)(sys ? 2 : 0) * g.Ny * ps + p) + part;
#pragma unroll 8
  for (int r = h.up; r < ny + 3; r += 2) {
    const double q = cv * vo[r * 64] + ce * eo[r * 64];
    out[(size_t)r * rs] = div_by(q, k2, rk);
  }
}

// ------------------------------------------------------- initial flow rate --
__global__ __launch_bounds__(256) void k_flowrate(MeanArgs a) {
  extern __shared__ double sm[];
  const Geom g = a.g;
  const int Ny = g.Ny, ny = g.ny;
  const size_t ps = g.ps, pstride = (size_t)Ny * ps;
  double *ur = sm, *wr = sm + Ny, *yy = sm + 2 * Ny, *red = sm + 3 * Ny;
  for (int i = threadIdx.x; i < Ny; i += blockDim.x) {
    ur[i] = a.V[(size_t)i * ps + g.nz].x;
    wr[i] = a.V[2 * pstride + (size_t)i * ps + g.nz].x;
    yy[i] = a.y[i];
  }
  __syncthreads();
  double fr[2];
  yintegr_block<2>(yy, sm, Ny, ny, red, fr);
  if (threadIdx.x == 0) {
    DevScalars *sc = a.sc;
    sc->fr[0] = fr[0];
    sc->fr[1] = fr[1];
    sc->fr[2] = 0.0;
    if (a.cpi) {
      if (a.cpi_type == 0)
        sc->meanpx = (1 - a.gamma) * 6 * a.ni / sc->fr[0];
      else
        sc->meanpx = (1.5 / a.gamma) * sc->fr[0] * a.ni;
    }
  }
}

// ------------------------------------------------------------ launchers --
// LDS of k_solve_lds: the columns of both systems with the tables, and the
// lower factors
static size_t solve_lds_columns(const Geom &g) {
  return ((size_t)2 * (g.ny + 3) * 64 + (size_t)(g.ny - 1) * SROW) * sizeof(double);
}
static size_t solve_lds_factors(const Geom &g) { return (size_t)2 * (g.ny - 1) * 16 * sizeof(double2); }
constexpr size_t LDS_MAX = 160 * 1024;

// The LDS kernel wherever its columns fit: the margin shrinks as the grid grows
// (3.7x at 31x64x31, 1.3x at 191x128x189, nine rounds of blocks) but stays.
bool solve_in_lds(const Geom &g) {
  return solve_lds_columns(g) <= LDS_MAX;
}

size_t solve_factors(const Geom &g) {
  if (solve_lds_columns(g) + solve_lds_factors(g) <= LDS_MAX) return 0;
  return (size_t)2 * (g.ny - 1) * group_stride(g.Nx * (g.nz + 1));
}

hipError_t launch_solve_lds(hipStream_t st, const SolveArgs &a, const UwArgs &u) {
  const Geom &g = a.g;
  const int blocks = (g.Nx * (g.nz + 1) + 1 + 15) / 16;
  dim3 grid((unsigned)((blocks + 7) / 8 * 8));
  const size_t all = solve_lds_columns(g) + solve_lds_factors(g);
  if (all <= LDS_MAX)
    hipLaunchKernelGGL(k_solve_lds<true>, grid, dim3(256), all, st, a, u, u.tab);
  else
    hipLaunchKernelGGL(k_solve_lds<false>, grid, dim3(256), solve_lds_columns(g), st, a, u, u.tab);
  return hipGetLastError();
}

hipError_t launch_solve(hipStream_t st, const SolveArgs &a) {
  const size_t lanes = (size_t)4 * (a.g.Nx * (a.g.nz + 1) + 1);
  dim3 grid(xcd_grid(lanes), 2);
  if (2 * lanes >= (size_t)12 * 64 * a.g.ncu)  // k_solve_ve_wide
    hipLaunchKernelGGL(k_solve_ve_wide, grid, dim3(256), 0, st, a, a.der);
  else
    hipLaunchKernelGGL(k_solve_ve, grid, dim3(256), 0, st, a, a.der);
  return hipGetLastError();
}
hipError_t launch_mean(hipStream_t st, const MeanArgs &a) {
  hipLaunchKernelGGL(k_mean, dim3(1), dim3(256), sizeof(double) * (4 * a.g.Ny + 3 * 256), st, a);
  return hipGetLastError();
}
hipError_t launch_uw(hipStream_t st, const UwArgs &a) {
  hipLaunchKernelGGL(k_uw, dim3((unsigned)((2 * a.g.npair + UW_BLOCK - 1) / UW_BLOCK)), dim3(UW_BLOCK), 0, st, a, a.der,
                     a.d0fac);
  return hipGetLastError();
}
hipError_t launch_flowrate(hipStream_t st, const MeanArgs &a) {
  hipLaunchKernelGGL(k_flowrate, dim3(1), dim3(256), sizeof(double) * (3 * a.g.Ny + 2 * 256), st, a);
  return hipGetLastError();
}

}  // namespace chan
