// k_rhs.hip -- K4: right-hand sides of the v-eta formulation for every
// interior row and wavenumber pair (buildrhs, dnsdata.f90:611-673).
//
// With kx = al, kz = be, k2 = kx^2 + kz^2, the explicit terms of the D2v and
// eta equations (:637-661) are stencils of four combinations of the products,
// formed once per row and pair:
//   G1 = k2 vv - kx^2 uu - 2 kx kz uw - kz^2 ww,  G2 = i kx uv + i kz vw
//   G3 = kx kz (uu - ww) + (kz^2 - kx^2) uw,      G4 = i kx vw - i kz uv
// which hold uu, vv and ww only as a = uu - ww and b = vv - ww: G1 = k2 b - kx^2 a
// - 2 kx kz uw, G3 = kx kz a + (kz^2 - kx^2) uw.
//   D2v: D1(G1) + D2(G2) + k2 D0(G2),             eta: D0(G3) + D1(G4)
// (the (0,0) mode's eta slot carries the mean flow: G4 = -(Re uv + i Re vw)).
// The implicit operators OS/SQ (:476-477) and the time derivative are one
// stencil of v and one of eta = i kz u - i kx w.
//
// One thread per (pair, chunk of rows) walks y and adds each row, as it is
// read, to the sums of the five output rows whose stencils reach it: five
// complex sums per pending row (explicit and implicit part of each equation, and
// D2 v), 100 FP64 registers' worth, where a five-row window of the eight fields that
// are read would be 40 complex values.  It then finishes the oldest row with
// the CN-RK3 time scheme (:486), writes the new rhs and replaces the stored
// explicit term.  The stencil coefficients come transposed (row r's weights
// in the five rows r-2..r+2), wave-uniform through the scalar cache.
//
// D2 v has a sum of its own because its terms nearly cancel: with its weights merged
// into those of the implicit part, which are rounded one by one, the right-hand side
// was up to twice and v after the solve up to three times as far from a 64-bit
// one (384 rows: 1.0e-15 for 3.3e-16).  The sum costs no time (191x384x189 1.10 ms,
// 1.14 without it).
//
// A body force enters the same sums as it is formed from F = F0 + gain * V_src
// (:643-659): D1(-i kx F_u - i kz F_w) and -k2 D0(F_v) in the D2v equation,
// D0(i kz F_u - i kx F_w) in the eta equation.  Its wall treatment (:616-628:
// F zero on the wall rows, ghost rows that make the compact D4 of the first
// and last interior rows vanish) is in the weights: the force has a table of
// its own, in which the ghost row is eliminated from rows 1 and ny-1 and the
// rows outside 1..ny-1 weigh nothing.  A feedback force reads only its gains
// besides what the right-hand side reads anyway: against force terms formed
// by a kernel of their own and read back, 34 for 155 us per substep at
// 63x96x47, 1.19 for 2.23 ms at 191x384x189.
//
// Bound by HBM and the memory-side cache on large grids: at 191x384x189 (FP64)
// 1.10 ms with five product fields, 7.0 GB of counted traffic at 6.3 TB/s (1.21
// with six, where a five-row window of the nine fields in two waves per SIMD and
// 48-row chunks took 1.39); by the length of the walk on small ones (31x64x31:
// 11.3 us, 61 before).
#include "chan_internal.hpp"

namespace chan {

// ghost rows of the body force (dnsdata.f90:617-628): with F(0) = F(-1) = 0 the
// compact D4 of row 1 is d4(0)F(1) + d4(1)F(2) + d4(2)F(3), and
// F(-1) = -D4 / d4(-2); at the top F(ny+1) = -D4 / d4(2) of row ny-1.
__device__ __forceinline__ cx<double> ghost_lo(const double *d4, cx<double> f1, cx<double> f2, cx<double> f3) {
  const cx<double> s = add(add(scl(d4[2], f1), scl(d4[3], f2)), scl(d4[4], f3));
  return cx<double>{-s.x / d4[0], -s.y / d4[0]};
}
__device__ __forceinline__ cx<double> ghost_hi(const double *d4, cx<double> f3, cx<double> f2, cx<double> f1) {
  const cx<double> s = add(add(scl(d4[0], f3), scl(d4[1], f2)), scl(d4[2], f1));
  return cx<double>{-s.x / d4[4], -s.y / d4[4]};
}

// F_c at interior row r (1 <= r <= ny-1) of pair p: the static part plus the
// feedback gain times the source velocity component.
__device__ __forceinline__ cx<double> force_at(const ForceArgs &a, int c, int s, int r, int p, int col) {
  const Geom &g = a.g;
  const size_t pstride = (size_t)g.Ny * g.ps, off = (size_t)(r + 1) * g.ps + p;
  cx<double> f = {0.0, 0.0};
  if (a.F0) f = a.F0[c * pstride + off];
  if (s >= 0) f = add(f, scl(a.gain[((size_t)c * g.Ny + (r + 1)) * (g.Nz + 1) + col], a.V[s * pstride + off]));
  return f;
}

// F of row r with the wall rows of buildrhs: zero on rows 0 and ny, ghost
// rows -1 and ny+1 from the compact D4 of rows 1 and ny-1.
__device__ __forceinline__ cx<double> force_row(const ForceArgs &a, const double *der, int c, int s, int r, int p,
                                                int col) {
  const int ny = a.g.ny;
  if (r >= 1 && r <= ny - 1) return force_at(a, c, s, r, p, col);
  if (r == -1) return ghost_lo(der + 15, force_at(a, c, s, 1, p, col), force_at(a, c, s, 2, p, col), force_at(a, c, s, 3, p, col));
  if (r == ny + 1)
    return ghost_hi(der + (size_t)(ny - 2) * 20 + 15, force_at(a, c, s, ny - 3, p, col), force_at(a, c, s, ny - 2, p, col),
                    force_at(a, c, s, ny - 1, p, col));
  return cx<double>{0.0, 0.0};
}

// one-wave blocks: each lane walks a row chunk, and smaller blocks spread the
// waves more evenly over the CUs
constexpr int RHS_BLOCK = 64;

// RD: the previous explicit terms enter (ode2 != 0); the first RK3 substep
// has ode2 = 0 and does not read them.
template <typename R, bool FORCE, bool RD>
__global__ __launch_bounds__(RHS_BLOCK) void k_rhs(RhsArgs<R> a, ForceArgs fa, const double *__restrict__ derT,
                                                   const double *__restrict__ derF, const DevScalars *__restrict__ sc) {
  // derT, derF and sc are separate restrict arguments so that their
  // wave-uniform values come through the scalar cache instead of vector
  // registers.
  const Geom g = a.g;
  const int p = blockIdx.x * RHS_BLOCK + threadIdx.x;
  if (p >= g.npair) return;
  const int ix = p / g.Nz, iz = p % g.Nz - g.nz;
  const double al = g.alfa0 * ix, be = g.beta0 * iz;
  const double al2 = al * al, be2 = be * be, albe = al * be, k2 = al2 + be2;
  const int y0 = 1 + (int)blockIdx.y * a.chunk;
  if (y0 > g.ny - 1) return;
  const int y1 = min(g.ny - 1, y0 + a.chunk - 1);
  const size_t ps = g.ps, pstride = (size_t)g.Ny * ps;
  const bool mean = (ix == 0 && iz == 0);
  const int col = mean ? g.Nz : iz + g.nz;
  // weights of the implicit v stencil: rdt D2, a sum of its own with the table's
  // weights, and cA D2 + cB D0 + ni D4; of eta: cC D0 + ni D2
  const double rdt = a.ode0 / a.dt;
  const double cA = -2.0 * a.ni * k2, cB = k2 * (a.ni * k2 - rdt), cC = rdt - a.ni * k2;
  const size_t rs = (size_t)(g.ny - 1) * ps;  // component stride of old/rhs

  // the row being read; all loads are unconditional, with the row clamped
  cx<R> np[NPROD];
  cx<double> nv[3], nold[2] = {{0.0, 0.0}, {0.0, 0.0}};
  cx<double> nf[3];  // static force
  double ng[3];      // feedback gains
  auto load = [&](int r) {  // row r (its plane is r + 1)
    const size_t off = (size_t)(r + 1) * ps + p;
#pragma unroll
    for (int q = 0; q < NPROD; q++) np[q] = a.P[q * pstride + off];
#pragma unroll
    for (int c = 0; c < 3; c++) nv[c] = a.V[c * pstride + off];
    if constexpr (FORCE) {
#pragma unroll
      for (int c = 0; c < 3; c++) {
        nf[c] = fa.F0 ? fa.F0[c * pstride + off] : cx<double>{0.0, 0.0};
        ng[c] = fa.src[c] >= 0 ? fa.gain[((size_t)c * g.Ny + (r + 1)) * (g.Nz + 1) + col] : 0.0;
      }
    }
    if constexpr (RD) {  // explicit terms of the row that r completes
      const size_t o = (size_t)(max(r - 2, 1) - 1) * ps + p;
      const cx<R> oe = a.old[o], ov = a.old[rs + o];
      nold[0] = cx<double>{(double)oe.x, (double)oe.y};
      nold[1] = cx<double>{(double)ov.x, (double)ov.y};
    }
  };
  // sums of the pending rows r-2..r+2 (slot m = row r-2+m): explicit and
  // implicit parts of the D2v (v) and eta (e) equations
  cx<double> sev[5], siv[5], sdv[5], see[5], sie[5];
#pragma unroll
  for (int m = 0; m < 5; m++) sev[m] = siv[m] = sdv[m] = see[m] = sie[m] = cx<double>{0.0, 0.0};
  load(y0 - 2);
  for (int r = y0 - 2; r <= y1 + 2; r++) {
    const auto D = [](cx<R> v) { return cx<double>{(double)v.x, (double)v.y}; };
    const cx<double> pa = D(np[0]), pb = D(np[1]), uv = D(np[2]), vw = D(np[3]), uw = D(np[4]);
    const cx<double> u = nv[0], v = nv[1], w = nv[2], old_e = nold[0], old_v = nold[1];
    cx<double> F[3];
    if constexpr (FORCE) {
      // zero where nothing is to be read into the force, whatever F0 holds there
      const bool in = r >= 1 && r <= g.ny - 1;
#pragma unroll
      for (int c = 0; c < 3; c++) {
        F[c] = cx<double>{0.0, 0.0};
        if (in) {
          F[c] = nf[c];
          const int s = fa.src[c];
          if (s >= 0) F[c] = add(F[c], scl(ng[c], s == 0 ? u : (s == 1 ? v : w)));
        }
      }
    }
    load(min(r + 1, g.ny + 1));
    cx<double> G1, G2, G3, G4, eta;
    G1.x = k2 * pb.x - al2 * pa.x - 2.0 * albe * uw.x;
    G1.y = k2 * pb.y - al2 * pa.y - 2.0 * albe * uw.y;
    G2 = cx<double>{-(al * uv.y + be * vw.y), al * uv.x + be * vw.x};
    G3.x = albe * pa.x + (be2 - al2) * uw.x;
    G3.y = albe * pa.y + (be2 - al2) * uw.y;
    G4 = cx<double>{be * uv.y - al * vw.y, al * vw.x - be * uv.x};
    eta = cx<double>{al * w.y - be * u.y, be * u.x - al * w.x};
    if (mean) {
      G4 = cx<double>{-uv.x, -vw.x};
      eta = cx<double>{u.x, w.x};
    }
    cx<double> H0, H1, H3;  // force terms: D0(H0) + D1(H1) in D2v, D0(H3) in eta
    if constexpr (FORCE) {
      H0 = cx<double>{-k2 * F[1].x, -k2 * F[1].y};
      H1 = cx<double>{al * F[0].y + be * F[2].y, -(al * F[0].x + be * F[2].x)};
      H3 = mean ? cx<double>{F[0].x, F[2].x} : cx<double>{al * F[2].y - be * F[0].y, be * F[0].x - al * F[2].x};
    }
    const double *df = derF + (size_t)(r + 1) * 10;  // [m][d0, d1]
    const double *d = derT + (size_t)(r + 1) * 20;  // [m][d0, d1, d2, d4]
#pragma unroll
    for (int m = 0; m < 5; m++) {
      const double d0 = d[4 * m], d1 = d[4 * m + 1], d2 = d[4 * m + 2], d4 = d[4 * m + 3];
      const double w2 = d2 + k2 * d0, wi = cA * d2 + cB * d0 + a.ni * d4, wj = cC * d0 + a.ni * d2;
      sev[m].x += d1 * G1.x + w2 * G2.x;
      sev[m].y += d1 * G1.y + w2 * G2.y;
      if constexpr (FORCE) {
        const double f0 = df[2 * m], f1 = df[2 * m + 1];
        sev[m].x += f0 * H0.x + f1 * H1.x;
        sev[m].y += f0 * H0.y + f1 * H1.y;
        see[m].x += f0 * H3.x;
        see[m].y += f0 * H3.y;
      }
      siv[m].x += wi * v.x;
      siv[m].y += wi * v.y;
      sdv[m].x += d2 * v.x;
      sdv[m].y += d2 * v.y;
      see[m].x += d0 * G3.x + d1 * G4.x;
      see[m].y += d0 * G3.y + d1 * G4.y;
      sie[m].x += wj * eta.x;
      sie[m].y += wj * eta.y;
    }
    const int iy = r - 2;  // complete now
    if (iy >= y0) {
      const size_t o = (size_t)(iy - 1) * ps + p;
      cx<double> ee = see[0];
      if (mean) {
        ee.x += sc->meanpx;
        ee.y += sc->meanpz;
      }
      cx<double> rv = {rdt * sdv[0].x + siv[0].x + a.ode1 * sev[0].x, rdt * sdv[0].y + siv[0].y + a.ode1 * sev[0].y};
      cx<double> re = {sie[0].x + a.ode1 * ee.x, sie[0].y + a.ode1 * ee.y};
      if constexpr (RD) {
        rv = sub(rv, scl(a.ode2, old_v));
        re = sub(re, scl(a.ode2, old_e));
      }
      a.rhs[rs + o] = rv;
      a.rhs[o] = re;
      if (a.store_old) {
        a.old[rs + o] = cx<R>{(R)sev[0].x, (R)sev[0].y};
        a.old[o] = cx<R>{(R)ee.x, (R)ee.y};
      }
    }
#pragma unroll
    for (int m = 0; m < 4; m++) {
      sev[m] = sev[m + 1];
      siv[m] = siv[m + 1];
      sdv[m] = sdv[m + 1];
      see[m] = see[m + 1];
      sie[m] = sie[m + 1];
    }
    sev[4] = siv[4] = sdv[4] = see[4] = sie[4] = cx<double>{0.0, 0.0};
  }
}

// The body force that buildrhs applies to the resident field, wall rows and
// ghost rows included, in the device layout (one thread per pair and
// component).
__global__ __launch_bounds__(256) void k_force(ForceArgs a, const double *__restrict__ der) {
  const Geom g = a.g;
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= g.npair) return;
  const int c = blockIdx.y;
  const int ix = p / g.Nz, iz = p % g.Nz - g.nz;
  const int col = (ix == 0 && iz == 0) ? g.Nz : iz + g.nz;
  cx<double> *o = a.out + c * (size_t)g.Ny * g.ps + p;
  for (int r = -1; r <= g.ny + 1; r++) o[(size_t)(r + 1) * g.ps] = force_row(a, der, c, a.src[c], r, p, col);
}

// Blocks of `block` pairs along x of the grid, rounded up to a multiple of 8:
// blocks (x, y) and (x, y+1) then sit a multiple of 8 apart in dispatch order,
// so round-robin dispatch puts the neighbouring row chunks of one pair block
// on one XCD and the halo rows that both read come from its L2 (k_rhs 1.3%
// faster in FP64 at 191x384x189).  The extra blocks exit at once.
static unsigned pair_blocks(const Geom &g, int block) {
  return (unsigned)(((g.npair + block - 1) / block + 7) / 8 * 8);
}

hipError_t launch_force(hipStream_t st, const ForceArgs &a) {
  dim3 grid((unsigned)((a.g.npair + 255) / 256), 3);
  hipLaunchKernelGGL(k_force, grid, dim3(256), 0, st, a, a.der);
  return hipGetLastError();
}

// Rows per chunk.  Every chunk reads four rows of its neighbours again, so
// long chunks move least, but each is one serial walk: on small grids chunks
// are halved until two waves per CU walk (31x64x31: 11.8 us with 3 rows, 42.8
// with 48; 100x97x77: 67 us with 24, 99 with 96, 97 with 4).  From 1024
// blocks of pairs on, short chunks make the whole grid advance through y as
// one front, whose shared rows the memory-side cache still holds
// (191x384x189: 1.21 ms with 8 rows, 1.30 with 48 or 96; 191x128x189 418 and
// 445 us; 127x384x127, 510 blocks, 602 and 594 us, 578 with 96; with a body
// force 1.19 and 1.29 ms at 191x384x189; all with six product fields).
static int rhs_chunk(const Geom &g) {
  const int blocks = (g.npair + RHS_BLOCK - 1) / RHS_BLOCK;
  if (blocks >= 1024) return 8;
  int c = 96;
  while (c > 2 && blocks * ((g.ny - 1 + c - 1) / c) < 2 * g.ncu) c = (c + 1) / 2;
  return c;
}

template <typename R, bool FORCE>
static void start_rhs(dim3 grid, hipStream_t st, const RhsArgs<R> &a, const ForceArgs &f) {
  if (a.ode2 != 0.0)
    hipLaunchKernelGGL((k_rhs<R, FORCE, true>), grid, dim3(RHS_BLOCK), 0, st, a, f, a.derT, f.derF, a.sc);
  else
    hipLaunchKernelGGL((k_rhs<R, FORCE, false>), grid, dim3(RHS_BLOCK), 0, st, a, f, a.derT, f.derF, a.sc);
}

template <typename R>
hipError_t launch_rhs(hipStream_t st, const RhsArgs<R> &args, const ForceArgs *force) {
  RhsArgs<R> a = args;
  a.chunk = rhs_chunk(a.g);
  dim3 grid(pair_blocks(a.g, RHS_BLOCK), (unsigned)((a.g.ny - 1 + a.chunk - 1) / a.chunk));
  if (force)
    start_rhs<R, true>(grid, st, a, *force);
  else
    start_rhs<R, false>(grid, st, a, ForceArgs{});
  return hipGetLastError();
}

template hipError_t launch_rhs<double>(hipStream_t, const RhsArgs<double> &, const ForceArgs *);
template hipError_t launch_rhs<float>(hipStream_t, const RhsArgs<float> &, const ForceArgs *);

}  // namespace chan
