// k_fft.hip -- the convolution products of one RK3 substep as three kernels
// over all y planes (convolutions, dnsdata.f90:487-602):
//
//   K1 k_zinv : V(iy,iz,ix,c) -> zero-pad z to nzd, backward c2c FFT in z
//               (IFT, ffts.f90:93-96)  -> A[plane][c][zb][ix][ZB]
//   K2 k_xpass: per physical-z row: Hermitian c2r in x (RFT, zero modes
//               nx+1..nxd), CFL maximum, the products, r2c in x keeping
//               modes 0..nx (HFT), times `factor`       -> B[plane][q][zb][ix][ZB]
//   K3 k_zfwd : forward c2c FFT in z, keep modes -nz..nz (FFT + izd)
//                                                       -> P[q][plane][pair]
//
// Products.  Five fields stand for the reference's six: uu - ww, vv - ww, uv, vw,
// uw.  The v-eta right-hand sides do not change when one field is added to uu, vv
// and ww alike (the divergence of an isotropic stress is a gradient; the compact
// stencils keep this exactly, k_rhs.hip), so ww is taken out of all three: one
// sixth less to write, transform in z and read.
//
// Grids.  The physical grid is the reference's (fftFIT, sizes 2^k and 3*2^k) where
// the CFL maximum is taken over its points.  The kept modes of the products are
// the same sums on every grid of more than 3 nz points in z and 3 nx in x, so
// where no CFL is asked for, the smallest supported size that large is used in z:
// 9*2^k where it is smaller than fftFIT's (576 for 768, 288 for 384, 144 for 192).  In x
// only where rows of that length are the faster ones (alias_free_x).
//
// The reference's pencil transposes (zTOx / xTOz, mpi_transpose.f90:50-117)
// are the layout changes between K1/K2 and K2/K3: both sides move ZB*16
// contiguous bytes per x mode.  Two real x-transforms share one complex FFT
// (u+iv on the way in, product pairs on the way out).
#include "chan_internal.hpp"

namespace chan {

// ------------------------------------------------------------------- K1 --
// the z transforms are bound by HBM traffic; the padded split exchange keeps
// their LDS footprint small
constexpr int ZXCH = fft::XCH_PAD;

// A z block is 32 (FP32) or 64 (FP64) bytes per x mode, short for memory
// transactions: the z kernels stage through LDS, where the G x modes of a
// block form one contiguous run of G*ZB values per z block, and lanes move
// whole runs (a wave touches 4 runs of 128 or 256 bytes).
// team stride of the staging area (a 32-byte shift per team keeps the
// staged writes and reads free of LDS bank conflicts)
template <int NZ>
constexpr int stage_stride() {
  return NZ + 4;
}
// x modes per block of the z kernels, and its threads: 256, or 192 where the team
// size is 3*2^k (N = 9*2^k)
template <int NZ>
constexpr int zteams() {
  return (fft::plan_nine(NZ) ? 192 : 256) / fft::Plan<NZ>::T;
}
template <int NZ>
constexpr int zthreads() {
  return zteams<NZ>() * fft::Plan<NZ>::T;
}
// The blocks stage the real and the imaginary parts in two rounds through
// one real-valued area: half the LDS of whole complex values, which would
// hold an FP64 block to three waves per SIMD and an FP32 block to six (four
// and eight with the two rounds: the FP64 step 1.5% and the FP32 z kernels
// 4-9% faster)
template <int NZ>
constexpr int zbuf_reals() {
  constexpr int G = zteams<NZ>();
  constexpr int fftr = G * fft::lds_reals<NZ, ZXCH>();
  constexpr int stg = G * stage_stride<NZ>();
  return fftr > stg ? fftr : stg;
}

template <int NZ, typename R>
__global__ __launch_bounds__(zthreads<NZ>()) void k_zinv(const cx<double> *__restrict__ V, cx<R> *__restrict__ A,
                                              const cx<R> *__restrict__ tw, Geom g, int plane0) {
  using PL = fft::Plan<NZ>;
  constexpr int T = PL::T, E = PL::E, G = zteams<NZ>(), NT = zthreads<NZ>(), SP = stage_stride<NZ>();
  __shared__ __align__(16) R lds[zbuf_reals<NZ>()];
  const int team = threadIdx.x / T, t = threadIdx.x % T;
  const int nxg = (g.Nx + G - 1) / G;
  int b = blockIdx.x;
  const int xg = b % nxg;
  b /= nxg;
  const int c = b % 3, pl = b / 3;
  const int ix = xg * G + team;
  const bool act = ix < g.Nx;
  const cx<double> *col = V + ((size_t)c * g.Ny + (plane0 + pl)) * g.ps + (size_t)(act ? ix : 0) * g.Nz;
  cx<R> e[E];
#pragma unroll
  for (int s = 0; s < E; s++) {
    const int z = t + T * s;
    const int iz = z <= g.nz ? z + g.nz : (z >= NZ - g.nz ? z - NZ + g.nz : -1);
    cx<double> v = {0.0, 0.0};
    if (act && iz >= 0) v = col[iz];
    e[s] = cx<R>{(R)v.x, (R)v.y};
  }
  fft::fft_slots<NZ, +1, true, ZXCH>(e, lds + team * fft::lds_reals<NZ, ZXCH>(), tw, t);
  cx<R> *dst = A + (size_t)(pl * 3 + c) * NZ * g.Nx;
  const int ix0 = xg * G, nact = min(G, g.Nx - ix0);
  R out[2][E];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    __syncthreads();  // the transforms' exchanges, or the previous round's reads, are done
#pragma unroll
    for (int s = 0; s < E; s++) lds[team * SP + t + T * s] = h ? e[s].y : e[s].x;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < E; i++) {
      const int el = (int)threadIdx.x + NT * i;  // G*NZ = NT*E elements per block
      const int zb = el / (G * ZB), w = el % (G * ZB), tm = w / ZB, r = w % ZB;
      out[h][i] = lds[min(tm, nact - 1) * SP + zb * ZB + r];
    }
  }
#pragma unroll
  for (int i = 0; i < E; i++) {
    const int el = (int)threadIdx.x + NT * i;
    const int zb = el / (G * ZB), w = el % (G * ZB), tm = w / ZB;
    if (tm < nact) dst[((size_t)zb * g.Nx + ix0) * ZB + w] = cx<R>{out[0][i], out[1][i]};
  }
}

// ------------------------------------------------------------------- K2 --
// the x pass runs five transforms per row and is bound by their arithmetic
// and LDS exchanges: radix-12 first pass, whole-complex padded exchanges
// (measured fastest; 2 waves/SIMD either way, u, v, w stay live)
constexpr bool XBIG = true;
constexpr int XXCH = fft::XCH_CPLX | fft::XCH_PAD;

template <int NT>
__device__ __forceinline__ void block_max_atomic(double m, double *red, unsigned long long *out) {
  // a maximum that keeps a NaN
  auto mx = [](double c, double o) { return (o > c || o != o) ? o : c; };
  double r;
  if constexpr (NT % 64 == 0) {
    // within each wave by lane exchanges, then across the waves in LDS
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) m = mx(m, __shfl_xor(m, s, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    r = red[0];
#pragma unroll
    for (int w = 1; w < NT / 64; w++) r = mx(r, red[w]);
  } else {
    red[threadIdx.x] = m;
    __syncthreads();
#pragma unroll
    for (int n = NT; n > 1; n = (n + 1) / 2) {
      const int h = (n + 1) / 2;
      if ((int)threadIdx.x + h < n) red[threadIdx.x] = mx(red[threadIdx.x], red[threadIdx.x + h]);
      __syncthreads();
    }
    r = red[0];
  }
  // values are >= 0 or NaN, so their bit patterns order as unsigned
  // integers (NaN above +Inf above every finite value)
  if (threadIdx.x == 0)
    atomicMax(out + (blockIdx.x % CFL_SLOTS) * CFL_STRIDE, (unsigned long long)__double_as_longlong(r));
}

// Product pairs: fields 0 uu-ww, 1 vv-ww, 2 uv, 3 vw, 4 uw as the real and
// imaginary parts of three complex sequences.
template <typename R>
__device__ __forceinline__ cx<R> product_pair(const int pp, R u, R v, R w) {
  if (pp == 0) return cx<R>{u * u - w * w, u * v};
  if (pp == 1) return cx<R>{u * w, v * v - w * w};
  return cx<R>{v * w, R(0)};
}
__device__ constexpr int pair_first(int pp) { return pp == 0 ? 0 : (pp == 1 ? 4 : 3); }
__device__ constexpr int pair_second(int pp) { return pp == 0 ? 2 : 1; }

// x modes per thread of the x pass: nxd >= 3(nx+1)/2 bounds Nx by M/3
template <int E>
constexpr int xmodes() {
  return (E + 2) / 3;
}

// value of the team-mate holding element M-k of a transform in slot layout:
// for t > 0 it is lane T-t, slot E-1-s; for t = 0 the thread itself, slot
// (E-s) mod E.  Teams of one wavefront at most (the 128-lane teams of the
// 1536-point rows combine their modes in fs1536_mode instead).
template <int T, int E, int MO, typename R>
__device__ __forceinline__ void mirror_pairs(const cx<R> (&e)[E], cx<R> (&m)[MO], int t, int nmode) {
  static_assert(T <= 64, "mirror_pairs works within one wavefront");
  const int lane = (int)(threadIdx.x & 63);
  const int src = lane - t + ((T - t) % T);
#pragma unroll
  for (int s = 0; s < MO; s++) {
    if (s * T < nmode) {  // uniform across the team
      const cx<R> send = e[E - 1 - s];
      const R rx = __shfl(send.x, src, 64), ry = __shfl(send.y, src, 64);
      m[s] = t ? cx<R>{rx, ry} : e[(E - s) % E];
    }
  }
}

// teams per x-pass block: one per row of a z block, or one per row of half a
// z block (TB = 2).  The halves read 32 of each 64 contiguous bytes of the
// z-block interleave; they are numbered 8 blocks apart, so that round-robin
// dispatch over the 8 XCDs puts both on one XCD and its L2.  Half blocks
// serve the 1536-point rows, whose 128-lane teams hold 29 KB of LDS each in
// FP64: two blocks then share a CU and one block's barriers overlap the
// other's work (25% less time per launch than four-row blocks at
// 511x512x511).  FP64 768-point rows gain 2.5% from half blocks; FP32 ones
// lose 7%, and keep whole z blocks.
template <int M, typename R>
constexpr int xteams() {
  return (M == 1536 || (M == 768 && sizeof(R) == 8)) ? 2 : ZB;
}
// MO_: direct-mode slots per lane, xmodes<E>() or fewer when nx + 1 <= T MO_
// (the launcher picks 3 for 768-point rows of at most 192 modes): the
// compiler then knows the middle slots of every backward transform are zero
// and drops the loads, selects and outputs that would only handle them
// FULL: nx + 1 == T MO_ exactly (nx = 191 for 768-point rows), so the mode
// bounds are compile-time constants and their selects and branches fold away
template <int M, typename R, bool PRODUCTS, int MO_ = xmodes<fft::Plan<M>::E>(), bool FULL = false>
__global__ __launch_bounds__((xteams<M, R>() * fft::Plan<M>::T), 2) void k_xpass(const cx<R> *__restrict__ A, cx<R> *__restrict__ B,
                                                                const cx<R> *__restrict__ tw, Geom g, int plane0,
                                                                int cfl_on, const double *__restrict__ dy, double dx,
                                                                double dz, R factor, unsigned long long *__restrict__ cfl_max,
                                                                int nplanes) {
  using PL = fft::Plan<M>;
  constexpr int TB = xteams<M, R>();
  constexpr int T = PL::T, E = PL::E, NT = TB * T;
  constexpr int MO = MO_;
  // FP64 768-point rows run their transforms in interleaved pairs
  // (fs768_bwd2 / fs768_fwd2): at two waves per SIMD the single transforms
  // leave the VALU waiting on their LDS exchanges
  constexpr bool ILV = M == 768 && sizeof(R) == 8;
  static_assert(MO <= xmodes<E>() && 2 * MO <= E, "direct and mirrored slots");
  // 768-point rows use the four-step transform (fs768_bwd/fwd), 1536-point
  // rows its two-wave form (fs1536_bwd/fwd); the samples between the two
  // directions sit in a permuted layout, which the pointwise CFL and products
  // do not see
  constexpr bool FS = M == 768, FS2 = M == 1536;
  constexpr int TEAM_R = FS ? 2 * fft::FS_LDS : (FS2 ? 4 * fft::FS_LDS : fft::lds_reals<M, XXCH>());
  static_assert(!FS2 || (T == 128 && E == 12 && MO == 4), "the two-wave 1536 transform needs 128-lane teams");
  __shared__ __align__(16) R fl[TB * TEAM_R];
  __shared__ double red[NT % 64 == 0 ? NT / 64 : NT];
  const int Nx = g.Nx, nx = FULL ? fft::Plan<M>::T * MO_ - 1 : g.nx, NZB = g.nzd / ZB;
  const int tid = threadIdx.x, t = tid % T;
  int zb, pl, zi;
  if constexpr (TB < ZB) {
    // half z blocks: the halves of tile 8q + x are blocks 16q + x and
    // 16q + 8 + x, which round-robin dispatch puts on one XCD
    static_assert(TB * 2 == ZB, "half z blocks");
    const int b = blockIdx.x, half = (b >> 3) & 1, tile = ((b >> 4) << 3) | (b & 7);
    if (tile >= NZB * nplanes) return;  // the whole block: padding of the grid
    zb = tile % NZB;
    pl = tile / NZB;
    zi = TB * half + tid / T;
  } else {
    zb = blockIdx.x % NZB;
    pl = blockIdx.x / NZB;
    zi = tid / T;
  }
  const int iy = plane0 + pl - 1;
  R *fr = fl + (tid / T) * TEAM_R;
  cx<R> *frc = reinterpret_cast<cx<R> *>(fr);

  // twiddles in LDS: their reads then wait on the LDS counter, not behind
  // the row loads still in flight on the vector-memory counter.  The
  // 768-point rows need only three table entries per lane, which they read
  // from global memory before their row loads: no staging and no block
  // barrier before the loads are issued.
  constexpr int NTW = FS ? 0 : (FS2 ? fft::FS2_TW : fft::plan_tw_size(M, XBIG));
  __shared__ __align__(16) cx<R> twl[NTW > 0 ? NTW : 1];
  if constexpr (NTW > 0) {
    for (int i = tid; i < NTW; i += NT) twl[i] = tw[i];
    __syncthreads();
  }
  // the four-step transform's twiddle powers, shared by the row's five transforms
  fft::FsTw<R> fw;
  if constexpr (FS)
    fw = fft::fs_twiddles(tw, t & 63);
  else if constexpr (FS2)
    fw = fft::fs_twiddles(twl, t & 63);
  auto bwd = [&](cx<R>(&v)[E]) {
    if constexpr (FS)
      fft::fs768_bwd<R, MO <= 3>(v, frc, fw, t);
    else if constexpr (FS2)
      fft::fs1536_bwd(v, frc, fw, twl, t);
    else
      fft::fft_slots<M, +1, XBIG, XXCH>(v, fr, twl, t);
  };
  auto fwd = [&](cx<R>(&v)[E]) {
    if constexpr (FS)
      fft::fs768_fwd(v, frc, fw, t);
    else if constexpr (FS2)
      fft::fs1536_fwd(v, frc, fw, t);
    else
      fft::fft_slots<M, -1, XBIG, XXCH>(v, fr, twl, t);
  };

  // Hermitian extension of row zi to M points: slot s holds mode k = t+T*s
  // (k <= nx) or the conjugate of mode M-k (k >= M-nx); Im of mode 0 is
  // dropped as c2r does.  Teams of at most one wavefront load only the
  // direct modes (slots s < MO, clamped in-row indices, all loads in flight
  // together) and take the mirrored ones from the partner lane: mode M-k of
  // lane t > 0 sits in slot E-1-s of lane T-t, lane 0 holds it in slot E-s.
  // Wider teams load both.
  constexpr bool SHFL = T <= 64;
  auto load_direct = [&](int c, cx<R>(&r)[MO]) {
    const cx<R> *src = A + ((size_t)(pl * 3 + c) * NZB + zb) * Nx * ZB + zi;
#pragma unroll
    for (int s = 0; s < MO; s++) r[s] = T * s <= nx ? src[(size_t)min(t + T * s, nx) * ZB] : cx<R>{0, 0};
  };
  auto extend = [&](const cx<R>(&r)[MO], cx<R>(&e)[E]) {
    const int lane = (int)(threadIdx.x & 63);
    const int src = lane - t + ((T - t) % T);
#pragma unroll
    for (int s = 0; s < E; s++) {
      const int k = t + T * s;
      cx<R> val = {0, 0};
      if (s < MO) {
        val = r[s < MO ? s : 0];
        if (k > nx) val = cx<R>{0, 0};
        if (k == 0) val.y = 0;
      }
      if (s >= E - MO) {
        const int sm = E - 1 - s;
        const R px = __shfl(r[sm].x, src, 64), py = __shfl(r[sm].y, src, 64);
        cx<R> mv = cx<R>{px, py};
        if (t == 0) mv = (E - s < MO) ? r[(E - s < MO) ? E - s : 0] : cx<R>{0, 0};
        if (k >= M - nx) val = cx<R>{mv.x, -mv.y};
      }
      e[s] = val;
    }
  };
  auto load_raw = [&](int c, cx<R>(&e)[E]) {
    const cx<R> *src = A + ((size_t)(pl * 3 + c) * NZB + zb) * Nx * ZB + zi;
#pragma unroll
    for (int s = 0; s < E; s++) {
      if (T * s > nx && T * s + T - 1 < M - nx) {
        e[s] = cx<R>{0, 0};
      } else {
        const int k = t + T * s;
        const int m = k <= nx ? k : (k >= M - nx ? M - k : 0);
        e[s] = src[(size_t)m * ZB];
      }
    }
  };
  auto fix_ext = [&](cx<R>(&e)[E]) {
#pragma unroll
    for (int s = 0; s < E; s++) {
      const int k = t + T * s;
      cx<R> v = e[s];
      if (k == 0) v.y = 0;
      if (k > nx) {
        if (k >= M - nx)
          v.y = -v.y;
        else
          v = cx<R>{0, 0};
      }
      e[s] = v;
    }
  };

  R u[E], v[E], w[E];
  {
    cx<R> e[E], f[E];
    cx<R> rw[SHFL ? MO : 1];
    if constexpr (SHFL) {
      cx<R> ru[MO], rv[MO];
      load_direct(0, ru);
      load_direct(1, rv);
      load_direct(2, rw);  // in flight during the first transform
      extend(ru, e);
      extend(rv, f);
    } else {
      load_raw(0, e);
      load_raw(1, f);
      fix_ext(e);
      fix_ext(f);
    }
#pragma unroll
    for (int s = 0; s < E; s++) e[s] = cx<R>{e[s].x - f[s].y, e[s].y + f[s].x};  // U + iV
    if constexpr (ILV) {
      extend(rw, f);
      fft::fs768_bwd2<R, MO <= 3>(e, f, frc, fw, t);
    } else {
      if constexpr (!SHFL) load_raw(2, f);  // in flight during the first transform
      bwd(e);
      if constexpr (SHFL)
        extend(rw, f);
      else
        fix_ext(f);
      bwd(f);
    }
#pragma unroll
    for (int s = 0; s < E; s++) {
      u[s] = e[s].x;
      v[s] = e[s].y;
      w[s] = f[s].x;
    }
  }

  // CFL maximum over the interior planes (dnsdata.f90:552-556).  FP64 gives
  // the reference's quotients (div_by: the correctly rounded divisions from
  // three reciprocals per row; its NaN for an infinite sample is reported as
  // the CFL check reports Inf); the split mode, whose samples are FP32,
  // multiplies by the reciprocals (within an FP64 rounding of the quotients).
  if (cfl_on && iy >= 1 && iy <= g.ny - 1) {
    const double dyv = dy[iy];
    const double rx = 1.0 / dx, ry = 1.0 / dyv, rz = 1.0 / dz;
    double m = 0.0;
    if constexpr (sizeof(R) == 4) {
#pragma unroll
      for (int s = 0; s < E; s++) {
        const double c = fabs((double)u[s]) * rx + fabs((double)v[s]) * ry + fabs((double)w[s]) * rz;
        m = (c > m || c != c) ? c : m;
      }
    } else {
#pragma unroll
      for (int s = 0; s < E; s++) {
        const double c = div_by(fabs((double)u[s]), dx, rx) + div_by(fabs((double)v[s]), dyv, ry) +
                         div_by(fabs((double)w[s]), dz, rz);
        m = (c > m || c != c) ? c : m;
      }
    }
    block_max_atomic<NT>(m, red, cfl_max);
  }

  if constexpr (PRODUCTS) {
    // pairs (uu-ww, uv) and (uw, vv-ww) share one forward transform each, vw has
    // its own; in this order u is dead once the second pair is formed, and v and
    // w once vw is
    auto form = [&](const int pp, cx<R>(&e)[E]) {
#pragma unroll
      for (int s = 0; s < E; s++) e[s] = product_pair(pp, u[s], v[s], w[s]);
    };
    // A_k = (Z_k + conj Z_{M-k})/2, B_k = (Z_k - conj Z_{M-k})/(2i), k=0..nx,
    // with the transform's normalisation factor applied here, once per mode
    auto emit = [&](const int pp, const cx<R>(&e)[E]) {
      cx<R> *da = B + ((size_t)(pl * NPROD + pair_first(pp)) * NZB + zb) * Nx * ZB + zi;
      cx<R> *db = B + ((size_t)(pl * NPROD + pair_second(pp)) * NZB + zb) * Nx * ZB + zi;
      const R hf = R(0.5) * factor;
      auto put = [&](int k, cx<R> z, cx<R> q) {
        if (pp == 2) {  // a real sequence alone
          da[(size_t)k * ZB] = cx<R>{z.x * factor, z.y * factor};
          return;
        }
        da[(size_t)k * ZB] = cx<R>{(z.x + q.x) * hf, (z.y - q.y) * hf};
        db[(size_t)k * ZB] = cx<R>{(z.y + q.y) * hf, (q.x - z.x) * hf};
      };
      if constexpr (FS2) {
        // wave h forms the modes 256 h .. 256 h + 255 (nx < 512 when M = 1536)
        const int h = t >> 6, tl = t & 63;
#pragma unroll
        for (int s = 0; s < MO; s++) {
          const int k = 256 * h + tl + 64 * s;
          if (k <= nx) {
            cx<R> z, q;
            fft::fs1536_mode(frc, twl, k, z, q);
            put(k, z, q);
          }
        }
        fft::team_sync<T>();  // the rows are the next transform's exchange area
      } else {
        cx<R> mz[MO];
        if (pp < 2) mirror_pairs<T, E, MO, R>(e, mz, t, nx + 1);
#pragma unroll
        for (int s = 0; s < MO; s++) {
          const int k = t + T * s;
          if (k <= nx) put(k, e[s], mz[s]);
        }
      }
    };
    if constexpr (ILV) {
      // the first pair alone while u, v, w are live, then the other two
      // together
      {
        cx<R> e[E];
        form(0, e);
        fwd(e);
        emit(0, e);
      }
      cx<R> e[E], f[E];
      form(1, e);
      form(2, f);
      fft::fs768_fwd2(e, f, frc, fw, t);
      emit(1, e);
      emit(2, f);
    } else {
#pragma unroll
      for (int pp = 0; pp < 3; pp++) {
        cx<R> e[E];
        form(pp, e);
        fwd(e);
        emit(pp, e);
      }
    }
  }
}

// ------------------------------------------------------------ K2, 9*2^k --
// The x pass of rows of 72, 144 and 288 points (no CFL): a block of 192 threads holds RW
// rows in teams of T = M/12 lanes, which straddle the wavefronts, so that the block
// synchronises as a whole; four rows are a z block.  As it does so anyway, it
// moves its global data through the teams' exchange areas: thread (mode, row) of
// a whole run reads and writes contiguous memory, the Hermitian extension and the
// mode split read their partners from LDS.
//
// Bound by the latency of its exchanges and barriers, at three waves per SIMD in FP64 (14
// spilled registers at 288 points).  us, against k_xpass on rows of 384 and 192 points
// of the same z grid: 95x128x95 166 for 188, 47x128x95 66 for 80; FP32 88 for 100,
// 40 for 42.
template <int M>
constexpr int xrows() {
  return 192 / fft::Plan<M>::T < ZB ? ZB : 192 / fft::Plan<M>::T;
}
template <int M, typename R>
__global__ __launch_bounds__((xrows<M>() * fft::Plan<M>::T), (sizeof(R) == 8 ? 3 : 4)) void k_xpass_blk(
    const cx<R> *__restrict__ A, cx<R> *__restrict__ B, const cx<R> *__restrict__ tw, Geom g, R factor, int nplanes) {
  using PL = fft::Plan<M>;
  constexpr int T = PL::T, E = PL::E, RW = xrows<M>(), NT = RW * T, MO = xmodes<E>(), MM = T * MO;  // MM modes at most
  constexpr int ROW = fft::xch_len<M, fft::XCH_PAD>();  // complex values of a row's area; 3 MM <= M
  constexpr int NTW = fft::plan_tw_size(M, true), ZPB = RW / ZB;  // twiddles, z blocks per block
  __shared__ __align__(16) cx<R> lds[RW * ROW];
  __shared__ __align__(16) cx<R> twl[NTW > 0 ? NTW : 1];
  const int Nx = g.Nx, nx = g.nx, NZB = g.nzd / ZB, ntile = NZB * nplanes;
  const int tid = threadIdx.x, t = tid % T, team = tid / T;
  cx<R> *mine = lds + team * ROW;
  R *fr = reinterpret_cast<R *>(mine);
  for (int i = tid; i < NTW; i += NT) twl[i] = tw[i];
  // modes 0..nx of u, v, w of every row: [row][c][MM]
  for (int zz = 0; zz < ZPB; zz++) {
    const int z = min((int)blockIdx.x * ZPB + zz, ntile - 1), pl = z / NZB, zb = z % NZB;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const cx<R> *src = A + ((size_t)(pl * 3 + c) * NZB + zb) * Nx * ZB;
      cx<R> *dst = lds + zz * ZB * ROW + c * MM;
#pragma unroll
      for (int j = 0; j < (ZB * MM + NT - 1) / NT; j++) {
        const int i = tid + NT * j;
        if (i < ZB * Nx) dst[(i % ZB) * ROW + i / ZB] = src[i];
      }
    }
  }
  __syncthreads();
  R u[E], v[E], w[E];
  {
    cx<R> e[E], f[E];
#pragma unroll
    for (int s = 0; s < E; s++) {
      e[s] = f[s] = cx<R>{0, 0};
      if (s >= MO && s < E - MO) continue;
      const int k = t + T * s, m = s < MO ? k : M - k;
      if (m > nx) continue;
      cx<R> a = mine[m], b = mine[MM + m], c = mine[2 * MM + m];
      if (s >= MO) {
        a.y = -a.y;
        b.y = -b.y;
        c.y = -c.y;
      }
      if (k == 0) a.y = b.y = c.y = 0;  // as c2r does
      e[s] = cx<R>{a.x - b.y, a.y + b.x};  // U + iV
      f[s] = c;
    }
    __syncthreads();
    fft::fft_slots<M, +1, true, fft::XCH_CPLX | fft::XCH_PAD>(e, fr, twl, t);
    fft::fft_slots<M, +1, true, fft::XCH_CPLX | fft::XCH_PAD>(f, fr, twl, t);
#pragma unroll
    for (int s = 0; s < E; s++) {
      u[s] = e[s].x;
      v[s] = e[s].y;
      w[s] = f[s].x;
    }
  }
#pragma unroll
  for (int pp = 0; pp < 3; pp++) {
    cx<R> e[E];
#pragma unroll
    for (int s = 0; s < E; s++) e[s] = product_pair(pp, u[s], v[s], w[s]);
    fft::fft_slots<M, -1, true, fft::XCH_CPLX | fft::XCH_PAD>(e, fr, twl, t);
    // the modes to LDS in natural order, then A_k = (Z_k + conj Z_{M-k})/2,
    // B_k = (Z_k - conj Z_{M-k})/(2i), k = 0..nx, times `factor`
#pragma unroll
    for (int s = 0; s < E; s++)
      if (s < MO || (pp < 2 && s >= E - MO)) mine[t + T * s] = e[s];
    __syncthreads();
    const R hf = R(0.5) * factor;
    for (int zz = 0; zz < ZPB; zz++) {
      const int z = (int)blockIdx.x * ZPB + zz, pl = z / NZB, zb = z % NZB;
      if (z >= ntile) break;
      cx<R> *da = B + ((size_t)(pl * NPROD + pair_first(pp)) * NZB + zb) * Nx * ZB;
      cx<R> *db = B + ((size_t)(pl * NPROD + pair_second(pp)) * NZB + zb) * Nx * ZB;
#pragma unroll
      for (int j = 0; j < (ZB * MM + NT - 1) / NT; j++) {
        const int i = tid + NT * j, k = i / ZB;
        if (i >= ZB * Nx) continue;
        const cx<R> *row = lds + (zz * ZB + i % ZB) * ROW;
        const cx<R> z0 = row[k];
        if (pp == 2) {
          da[i] = cx<R>{z0.x * factor, z0.y * factor};
        } else {
          const cx<R> q = row[k ? M - k : 0];
          da[i] = cx<R>{(z0.x + q.x) * hf, (z0.y - q.y) * hf};
          db[i] = cx<R>{(z0.y + q.y) * hf, (q.x - z0.x) * hf};
        }
      }
    }
    __syncthreads();
  }
}

// -------------------------------------------------------- K2, few rows --
// The x pass of short rows, whose teams of less than 16 lanes leave k_xpass's waves
// half empty, and of few rows: three teams per row, one for each field on the way
// in and one for each product pair on the way out, so that a row's chain is two
// transforms instead of five.  They meet in LDS: the samples and the products' modes
// of a z block's rows, which its threads then write out as whole runs.
//
// Bound by that chain where the rows are few: 15x32x15 (rows of 48) 8.9 for 13.0 us,
// 31x64x31 (96) 19.8 for 22.0, 23x64x31 (72) 18.8 for 23.4.
template <int M, typename R>
__global__ __launch_bounds__(3 * ZB * fft::Plan<M>::T) void k_xpass_few(const cx<R> *__restrict__ A, cx<R> *__restrict__ B,
                                                                        const cx<R> *__restrict__ tw, Geom g, int plane0,
                                                                        int cfl_on, const double *__restrict__ dy, double dx,
                                                                        double dz, R factor,
                                                                        unsigned long long *__restrict__ cfl_max) {
  using PL = fft::Plan<M>;
  constexpr int T = PL::T, E = PL::E, MO = xmodes<E>(), NT = 3 * ZB * T, XC = fft::XCH_CPLX | fft::XCH_PAD;
  constexpr int ROW = fft::xch_len<M, fft::XCH_PAD>(), NTW = fft::plan_tw_size(M, true);
  __shared__ __align__(16) cx<R> lds[3 * ZB * ROW];
  __shared__ __align__(16) cx<R> twl[NTW > 0 ? NTW : 1];
  __shared__ double red[NT];
  const int nx = g.nx, Nx = g.Nx, NZB = g.nzd / ZB, zb = blockIdx.x % NZB, pl = blockIdx.x / NZB, iy = plane0 + pl - 1;
  const int tid = threadIdx.x, t = tid % T, zi = tid / T % ZB, c = tid / (T * ZB);
  cx<R> *mine = lds + (c * ZB + zi) * ROW;
  R *fr = reinterpret_cast<R *>(mine);
  cx<R> e[E];
  {
    const cx<R> *src = A + ((size_t)(pl * 3 + c) * NZB + zb) * Nx * ZB + zi;
#pragma unroll
    for (int s = 0; s < E; s++) {
      e[s] = cx<R>{0, 0};
      if (s >= MO && s < E - MO) continue;
      const int k = t + T * s, m = s < MO ? k : M - k;
      if (m <= nx) e[s] = src[(size_t)m * ZB];
      if (s >= MO) e[s].y = -e[s].y;
      if (k == 0) e[s].y = 0;  // as c2r does
    }
  }
  for (int i = tid; i < NTW; i += NT) twl[i] = tw[i];
  __syncthreads();
  fft::fft_slots<M, +1, true, XC>(e, fr, twl, t);
#pragma unroll
  for (int s = 0; s < E; s++) fr[t + T * s] = e[s].x;
  __syncthreads();
  const R *u = reinterpret_cast<const R *>(lds + zi * ROW), *v = u + 2 * ZB * ROW, *w = v + 2 * ZB * ROW;
  // the CFL maximum as k_xpass takes it, a third of the samples per team
  if (cfl_on && iy >= 1 && iy <= g.ny - 1) {
    const double dyv = dy[iy];
    const double rx = 1.0 / dx, ry = 1.0 / dyv, rz = 1.0 / dz;
    double m = 0.0;
#pragma unroll
    for (int j = 0; j < (E + 2) / 3; j++) {
      const int n = t + T * (3 * j + c);
      if (n >= M) continue;
      const double au = fabs((double)u[n]), av = fabs((double)v[n]), aw = fabs((double)w[n]);
      const double q = sizeof(R) == 4 ? au * rx + av * ry + aw * rz
                                      : div_by(au, dx, rx) + div_by(av, dyv, ry) + div_by(aw, dz, rz);
      m = (q > m || q != q) ? q : m;
    }
    block_max_atomic<NT>(m, red, cfl_max);
  }
#pragma unroll
  for (int s = 0; s < E; s++) {
    const int n = t + T * s;
    const R a = u[n], b = v[n], d = w[n];
    e[s].x = c == 0 ? a * a - d * d : (c == 1 ? a * d : b * d);  // product_pair(c, a, b, d)
    e[s].y = c == 0 ? a * b : (c == 1 ? b * b - d * d : R(0));
  }
  __syncthreads();
  fft::fft_slots<M, -1, true, XC>(e, fr, twl, t);
#pragma unroll
  for (int s = 0; s < E; s++)
    if (s < MO || s >= E - MO) mine[t + T * s] = e[s];
  __syncthreads();
  const R hf = R(0.5) * factor;
  const int first = c == 0 ? pair_first(0) : (c == 1 ? pair_first(1) : pair_first(2));
  cx<R> *da = B + ((size_t)(pl * NPROD + first) * NZB + zb) * Nx * ZB;
  cx<R> *db = B + ((size_t)(pl * NPROD + pair_second(c)) * NZB + zb) * Nx * ZB;
#pragma unroll
  for (int j = 0; j < MO; j++) {
    const int i = zi * T + t + ZB * T * j, k = i / ZB;
    if (i >= ZB * Nx) continue;
    const cx<R> *row = lds + (c * ZB + i % ZB) * ROW;
    const cx<R> z0 = row[k];
    if (c == 2) {
      da[i] = cx<R>{z0.x * factor, z0.y * factor};
    } else {
      const cx<R> q = row[k ? M - k : 0];
      da[i] = cx<R>{(z0.x + q.x) * hf, (z0.y - q.y) * hf};
      db[i] = cx<R>{(z0.y + q.y) * hf, (q.x - z0.x) * hf};
    }
  }
}

// ------------------------------------------------------------------- K3 --
template <int NZ, typename R>
__global__ __launch_bounds__(zthreads<NZ>()) void k_zfwd(const cx<R> *__restrict__ B, cx<R> *__restrict__ P,
                                              const cx<R> *__restrict__ tw, Geom g, int plane0) {
  using PL = fft::Plan<NZ>;
  constexpr int T = PL::T, E = PL::E, G = zteams<NZ>(), NT = zthreads<NZ>(), SP = stage_stride<NZ>();
  __shared__ __align__(16) R lds[zbuf_reals<NZ>()];
  const int team = threadIdx.x / T, t = threadIdx.x % T;
  const int nxg = (g.Nx + G - 1) / G;
  int b = blockIdx.x;
  const int xg = b % nxg;
  b /= nxg;
  const int q = b % NPROD, pl = b / NPROD;
  const int ix = xg * G + team;
  const bool act = ix < g.Nx;
  const cx<R> *src = B + (size_t)(pl * NPROD + q) * NZ * g.Nx;
  cx<R> e[E];
  const int ix0 = xg * G, nact = min(G, g.Nx - ix0);
  cx<R> v[E];
#pragma unroll
  for (int i = 0; i < E; i++) {  // all loads in flight together, clamped into the block's runs
    const int el = (int)threadIdx.x + NT * i;
    const int zb = el / (G * ZB), w = el % (G * ZB);
    v[i] = src[((size_t)zb * g.Nx + ix0) * ZB + min(w, nact * ZB - 1)];
  }
#pragma unroll
  for (int h = 0; h < 2; h++) {
#pragma unroll
    for (int i = 0; i < E; i++) {
      const int el = (int)threadIdx.x + NT * i;
      const int zb = el / (G * ZB), w = el % (G * ZB), tm = w / ZB, r = w % ZB;
      lds[tm * SP + zb * ZB + r] = tm < nact ? (h ? v[i].y : v[i].x) : R(0);
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < E; s++) (h ? e[s].y : e[s].x) = lds[team * SP + t + T * s];
    __syncthreads();  // the next round and the transforms reuse the staging area
  }
  fft::fft_slots<NZ, -1, true, ZXCH>(e, lds + team * fft::lds_reals<NZ, ZXCH>(), tw, t);
  if (act) {
    cx<R> *dst = P + ((size_t)q * g.Ny + (plane0 + pl)) * g.ps + (size_t)ix * g.Nz;
#pragma unroll
    for (int s = 0; s < E; s++) {
      const int k = t + T * s;
      const int iz = k <= g.nz ? k + g.nz : (k >= NZ - g.nz ? k - NZ + g.nz : -1);
      if (iz >= 0) dst[iz] = e[s];
    }
  }
}

// ------------------------------------------------------------- selftest --
template <int N, int S>
__global__ __launch_bounds__(256) void k_fft_test(cx<double> *__restrict__ data, const cx<double> *__restrict__ tw,
                                                  int batch) {
  using PL = fft::Plan<N>;
  constexpr int T = PL::T, E = PL::E, G = 256 / T;
  __shared__ double lds[G * N];
  const int team = threadIdx.x / T, t = threadIdx.x % T;
  const int row = blockIdx.x * G + team;
  const bool act = row < batch;
  cx<double> *x = data + (size_t)(act ? row : 0) * N;
  cx<double> e[E];
#pragma unroll
  for (int s = 0; s < E; s++) e[s] = act ? x[t + T * s] : cx<double>{0, 0};
  fft::fft_slots<N, S>(e, lds + team * N, tw, t);
  if (act)
#pragma unroll
    for (int s = 0; s < E; s++) x[t + T * s] = e[s];
}

// ------------------------------------------------------ four-step test --
// Rows of 768 complex FP64 values in natural order.  sign +1: slot layout ->
// fs768_bwd -> written back in natural order through fs768_index; sign -1:
// read in layout P -> fs768_fwd -> natural order.  inner > 1 first runs
// inner-1 backward/forward pairs (for timing; the data grows by 768 per pair).
__global__ __launch_bounds__(256) void k_fs768_test(const cx<double> *__restrict__ in, cx<double> *__restrict__ out,
                                                    const cx<double> *__restrict__ tw, int batch, int sign, int inner) {
  __shared__ __align__(16) cx<double> lds[4 * fft::FS_LDS];
  __shared__ cx<double> twl[fft::FS_TW];
  for (int i = threadIdx.x; i < fft::FS_TW; i += 256) twl[i] = tw[i];
  __syncthreads();
  const int team = threadIdx.x / 64, t = threadIdx.x % 64;
  const int row = blockIdx.x * 4 + team;
  const bool act = row < batch;
  const cx<double> *x = in + (size_t)(act ? row : 0) * 768;
  cx<double> *L = lds + team * fft::FS_LDS;
  const fft::FsTw<double> fw = fft::fs_twiddles(twl, t);
  cx<double> e[12];
  if (sign > 0) {
#pragma unroll
    for (int s = 0; s < 12; s++) e[s] = x[t + 64 * s];
    for (int k = 1; k < inner; k++) {
      fft::fs768_bwd(e, L, fw, t);
      fft::fs768_fwd(e, L, fw, t);
    }
    fft::fs768_bwd(e, L, fw, t);
    if (act)
#pragma unroll
      for (int s = 0; s < 12; s++) out[(size_t)row * 768 + fft::fs768_index(t, s)] = e[s];
  } else {
#pragma unroll
    for (int s = 0; s < 12; s++) e[s] = x[fft::fs768_index(t, s)];
    for (int k = 1; k < inner; k++) {
      fft::fs768_fwd(e, L, fw, t);
      fft::fs768_bwd(e, L, fw, t);
    }
    fft::fs768_fwd(e, L, fw, t);
    if (act)
#pragma unroll
      for (int s = 0; s < 12; s++) out[(size_t)row * 768 + t + 64 * s] = e[s];
  }
}

hipError_t launch_fs768_test(const cx<double> *in, cx<double> *out, const cx<double> *tw, int batch, int sign, int inner) {
  hipLaunchKernelGGL(k_fs768_test, dim3((unsigned)((batch + 3) / 4)), dim3(256), 0, 0, in, out, tw, batch, sign, inner);
  return hipGetLastError();
}

// ------------------------------------------------------------- benchmark --
// out-of-place batched transforms for timing the exchange/plan variants:
// variants 0-7: bit 0 complex exchange, bit 1 padded exchange, bit 2 radix-4/3
// plan; 8-11: complex exchange padded every 16, 8, 4 elements, XOR layout
template <int N, int S, bool BIG, int XCH>
__global__ __launch_bounds__(256) void k_fft_bench(const cx<double> *__restrict__ in, cx<double> *__restrict__ out,
                                                   const cx<double> *__restrict__ tw, int batch, int inner) {
  using PL = fft::Plan<N, BIG>;
  constexpr int T = PL::T, E = PL::E, G = 256 / T, L = fft::lds_reals<N, XCH>();
  __shared__ __align__(16) double lds[G * L];
  const int team = threadIdx.x / T, t = threadIdx.x % T;
  const int row = blockIdx.x * G + team;
  const bool act = row < batch;
  const cx<double> *x = in + (size_t)(act ? row : 0) * N;
  cx<double> e[E];
#pragma unroll
  for (int s = 0; s < E; s++) e[s] = act ? x[t + T * s] : cx<double>{0, 0};
  for (int k = 0; k < inner; k++) fft::fft_slots<N, S, BIG, XCH>(e, lds + team * L, tw, t);
  if (act)
#pragma unroll
    for (int s = 0; s < E; s++) out[(size_t)row * N + t + T * s] = e[s];
}

template <int N, int S, bool BIG, int XCH>
hipError_t launch_bench_v(const cx<double> *in, cx<double> *out, const cx<double> *tw, int batch, int inner) {
  constexpr int G = 256 / fft::Plan<N, BIG>::T;
  hipLaunchKernelGGL((k_fft_bench<N, S, BIG, XCH>), dim3((unsigned)((batch + G - 1) / G)), dim3(256), 0, 0, in, out, tw,
                     batch, inner);
  return hipGetLastError();
}

template <int N, int S>
hipError_t launch_bench_n(int variant, const cx<double> *in, cx<double> *out, const cx<double> *tw, int batch, int inner) {
  switch (variant) {
    case 0: return launch_bench_v<N, S, true, 0>(in, out, tw, batch, inner);
    case 1: return launch_bench_v<N, S, true, 1>(in, out, tw, batch, inner);
    case 2: return launch_bench_v<N, S, true, 2>(in, out, tw, batch, inner);
    case 3: return launch_bench_v<N, S, true, 3>(in, out, tw, batch, inner);
    case 4: return launch_bench_v<N, S, false, 0>(in, out, tw, batch, inner);
    case 5: return launch_bench_v<N, S, false, 1>(in, out, tw, batch, inner);
    case 6: return launch_bench_v<N, S, false, 2>(in, out, tw, batch, inner);
    case 7: return launch_bench_v<N, S, false, 3>(in, out, tw, batch, inner);
    // complex exchanges with the timing layouts
    case 8: return launch_bench_v<N, S, true, fft::XCH_CPLX | fft::XCH_PAD16>(in, out, tw, batch, inner);
    case 9: return launch_bench_v<N, S, true, fft::XCH_CPLX | fft::XCH_PAD8>(in, out, tw, batch, inner);
    case 10: return launch_bench_v<N, S, true, fft::XCH_CPLX | fft::XCH_PAD4>(in, out, tw, batch, inner);
    case 11: return launch_bench_v<N, S, true, fft::XCH_CPLX | fft::XCH_XOR>(in, out, tw, batch, inner);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_fft_bench(int N, int sign, int variant, const cx<double> *in, cx<double> *out, const cx<double> *tw,
                            int batch, int inner) {
  switch (N) {
    case 384: return sign < 0 ? launch_bench_n<384, -1>(variant, in, out, tw, batch, inner) : launch_bench_n<384, 1>(variant, in, out, tw, batch, inner);
    case 768: return sign < 0 ? launch_bench_n<768, -1>(variant, in, out, tw, batch, inner) : launch_bench_n<768, 1>(variant, in, out, tw, batch, inner);
    case 1536: return sign < 0 ? launch_bench_n<1536, -1>(variant, in, out, tw, batch, inner) : launch_bench_n<1536, 1>(variant, in, out, tw, batch, inner);
  }
  return hipErrorInvalidValue;
}

// ------------------------------------------------------------ launchers --
#define CHAN_FOR_NINES_X(X) X(36) X(72) X(144) X(288)
#define CHAN_FOR_NINES(X) CHAN_FOR_NINES_X(X) X(576) X(1152)
#define CHAN_FOR_SIZES(X) X(12) X(24) X(48) X(96) X(192) X(384) X(768) X(1536) X(16) X(32) X(64) X(128) X(256) X(512) X(1024)

#define CHAN_FOR_FEW(X) X(12) X(24) X(48) X(96) X(16) X(32) X(64) X(128) X(36) X(72)
// sizes whose products k_xpass_few always forms: it does six transforms for five,
// but in full waves (31x128x31 28.9 for 34.5 us; 11x128x95, rows of 36 that
// k_xpass_blk could take, 26.5 for 32.8)
template <int M>
constexpr bool few_always() {
  return M == 36 || (M % 9 != 0 && fft::Plan<M>::T < 16);
}
// rows of 72 points fill k_xpass_blk's waves too: k_xpass_few has them while its
// blocks of two waves are all resident, at four waves per SIMD (23x64x31, 1608 blocks,
// 18.8 for 23.4 us; 23x128x95, 9432 blocks, 56.1 for 51.9)
static bool use_few(int M, unsigned ntile, int ncu) { return M != 72 || ntile <= 8u * (unsigned)ncu; }

template <typename R>
hipError_t launch_zinv(int NZ, hipStream_t st, const cx<double> *V, cx<R> *A, const cx<R> *tw, const Geom &g, int plane0,
                       int nplanes) {
  switch (NZ) {
#define X(N)                                                                              \
  case N: {                                                                               \
    constexpr int G = zteams<N>();                                                        \
    dim3 grid((unsigned)(((g.Nx + G - 1) / G) * 3 * nplanes));                            \
    hipLaunchKernelGGL((k_zinv<N, R>), grid, dim3(zthreads<N>()), 0, st, V, A, tw, g, plane0); \
    return hipGetLastError();                                                             \
  }
    CHAN_FOR_SIZES(X)
    CHAN_FOR_NINES(X)
#undef X
  }
  return hipErrorInvalidValue;
}

template <typename R>
hipError_t launch_xpass(int M, hipStream_t st, const cx<R> *A, cx<R> *B, const cx<R> *tw, const Geom &g, int plane0,
                        int nplanes, bool products, int cfl_on, const double *dy, double dx, double dz, R factor,
                        unsigned long long *cfl_max) {
  const unsigned ntile = (unsigned)((g.nzd / ZB) * nplanes);
  if (products && use_few(M, ntile, g.ncu)) switch (M) {
#define X(N)                                                                                                         \
  case N:                                                                                                            \
    hipLaunchKernelGGL((k_xpass_few<N, R>), dim3(ntile), dim3(3 * ZB * fft::Plan<N>::T), 0, st, A, B, tw, g, plane0, \
                       cfl_on, dy, dx, dz, factor, cfl_max);                                                         \
    return hipGetLastError();
      CHAN_FOR_FEW(X)
#undef X
    }
  switch (M) {
#define X(N)                                                                                                          \
  case N: {                                                                                                           \
    dim3 blk(xteams<N, R>() * fft::Plan<N>::T);                                                                       \
    dim3 grid(xteams<N, R>() < ZB ? 16 * ((ntile + 7) / 8) : ntile);                                                  \
    if constexpr (!few_always<N>()) {                                                                                 \
      if constexpr (N == 768) {                                                                                       \
        if (products && g.nx + 1 <= 192) {                                                                            \
          if (g.nx + 1 == 192)                                                                                        \
            hipLaunchKernelGGL((k_xpass<N, R, true, 3, true>), grid, blk, 0, st, A, B, tw, g, plane0, cfl_on, dy, dx, \
                               dz, factor, cfl_max, nplanes);                                                         \
          else                                                                                                        \
            hipLaunchKernelGGL((k_xpass<N, R, true, 3>), grid, blk, 0, st, A, B, tw, g, plane0, cfl_on, dy, dx, dz,   \
                               factor, cfl_max, nplanes);                                                             \
          return hipGetLastError();                                                                                   \
        }                                                                                                             \
      }                                                                                                               \
      if (products) {                                                                                                 \
        hipLaunchKernelGGL((k_xpass<N, R, true>), grid, blk, 0, st, A, B, tw, g, plane0, cfl_on, dy, dx, dz, factor,  \
                           cfl_max, nplanes);                                                                         \
        return hipGetLastError();                                                                                     \
      }                                                                                                               \
    }                                                                                                                 \
    hipLaunchKernelGGL((k_xpass<N, R, false>), grid, blk, 0, st, A, B, tw, g, plane0, cfl_on, dy, dx, dz, factor,     \
                       cfl_max, nplanes);                                                                             \
    return hipGetLastError();                                                                                         \
  }
    CHAN_FOR_SIZES(X)
#undef X
#define X(N)                                                                                                          \
  case N: {                                                                                                           \
    if (!products || cfl_on) break;                                                                                   \
    constexpr int RW = xrows<N>();                                                                                    \
    if constexpr (!few_always<N>())                                                                                   \
      hipLaunchKernelGGL((k_xpass_blk<N, R>), dim3((ntile + RW / ZB - 1) / (RW / ZB)), dim3(RW * fft::Plan<N>::T), 0, \
                         st, A, B, tw, g, factor, nplanes);                                                           \
    return hipGetLastError();                                                                                         \
  }
    CHAN_FOR_NINES_X(X)
#undef X
  }
  return hipErrorInvalidValue;
}

template <typename R>
hipError_t launch_zfwd(int NZ, hipStream_t st, const cx<R> *B, cx<R> *P, const cx<R> *tw, const Geom &g, int plane0,
                       int nplanes) {
  switch (NZ) {
#define X(N)                                                                         \
  case N: {                                                                          \
    constexpr int G = zteams<N>();                                                   \
    dim3 grid((unsigned)(((g.Nx + G - 1) / G) * NPROD * nplanes));                   \
    hipLaunchKernelGGL((k_zfwd<N, R>), grid, dim3(zthreads<N>()), 0, st, B, P, tw, g, plane0); \
    return hipGetLastError();                                                        \
  }
    CHAN_FOR_SIZES(X)
    CHAN_FOR_NINES(X)
#undef X
  }
  return hipErrorInvalidValue;
}

hipError_t launch_fft_test(int N, int sign, hipStream_t st, cx<double> *data, const cx<double> *tw, int batch) {
  switch (N) {
#define X(NN)                                                                                      \
  case NN: {                                                                                       \
    constexpr int G = 256 / fft::Plan<NN>::T;                                                      \
    dim3 grid((unsigned)((batch + G - 1) / G));                                                    \
    if (sign < 0)                                                                                  \
      hipLaunchKernelGGL((k_fft_test<NN, -1>), grid, dim3(256), 0, st, data, tw, batch);           \
    else                                                                                           \
      hipLaunchKernelGGL((k_fft_test<NN, +1>), grid, dim3(256), 0, st, data, tw, batch);           \
    return hipGetLastError();                                                                      \
  }
    CHAN_FOR_SIZES(X)
#undef X
  }
  return hipErrorInvalidValue;
}

// the smallest size of the form 9*2^k in [need, below), or `below` when none is
// (z).  Faster wherever the grid fills the chip, and the x pass has fewer rows; us, this and
// the physical size, z inverse and z forward: 191x384x189 (576 and 768 points) 646 and 758,
// 1090 and 1291; 383x48x383 (1152 and 1536) 329 and 400, 642 and 779, FP32 293 and 304, 403
// and 493; 15x24x383 15.5 and 18.3, 20.7 and 24.9.  Grids of one round of blocks lose up to a
// us on the inverse in FP32 (7x12x95, 288 and 384, 10.0 and 9.1) and gain it on the x pass (8.2
// and 9.1 with the CFL maximum).
int alias_free_z(int need, int below) {
#define X(N) \
  if (N >= need && N < below) return N;
  CHAN_FOR_NINES(X)
#undef X
  return below;
}
// The same for the rows of the x pass, of which there are `tiles` groups of ZB.  Rows of
// 576 and 1152 points lose to k_xpass's four-step rows of 768 and 1536 (us, same z
// grid: 191x384x189 1972 and 1687, FP32 994 and 822, 191x48x47 72 and 66, 383x48x95 438 and
// 328).  Rows of 144 and 288 need tiles enough for their larger blocks: four per CU
// (95x16x11, 171 tiles, 20.6 and 16.0; 95x24x23, 486, 21.8 and 21.6; 95x24x47, 972, 27.2
// and 28.8; 47x40x23, 774, 17.4 and 17.0; 47x40x47, 1548, 20.8 and 23.4), rows of 144 in FP32
// eight (1548 tiles 16.1 and 15.6, 2412 19.2 and 19.4).  Shorter rows have k_xpass_few.
int alias_free_x(int need, int below, unsigned tiles, int ncu, bool fp32) {
#define X(N)                                                                              \
  if (N >= need && N < below) {                                                           \
    const unsigned per_cu = N < 144 ? 0 : (N == 144 && fp32 ? 8 : 4);                     \
    return tiles >= per_cu * (unsigned)ncu ? N : below;                                   \
  }
  CHAN_FOR_NINES_X(X)
#undef X
  return below;
}

int fft_size_supported(int N) {
  switch (N) {
#define X(NN) case NN:
    CHAN_FOR_SIZES(X)
#undef X
    return 1;
  }
  return 0;
}

template hipError_t launch_zinv<double>(int, hipStream_t, const cx<double> *, cx<double> *, const cx<double> *,
                                        const Geom &, int, int);
template hipError_t launch_xpass<double>(int, hipStream_t, const cx<double> *, cx<double> *, const cx<double> *,
                                         const Geom &, int, int, bool, int, const double *, double, double, double,
                                         unsigned long long *);
template hipError_t launch_zfwd<double>(int, hipStream_t, const cx<double> *, cx<double> *, const cx<double> *,
                                        const Geom &, int, int);
template hipError_t launch_zinv<float>(int, hipStream_t, const cx<double> *, cx<float> *, const cx<float> *,
                                       const Geom &, int, int);
template hipError_t launch_xpass<float>(int, hipStream_t, const cx<float> *, cx<float> *, const cx<float> *,
                                        const Geom &, int, int, bool, int, const double *, double, double, float,
                                        unsigned long long *);
template hipError_t launch_zfwd<float>(int, hipStream_t, const cx<float> *, cx<float> *, const cx<float> *,
                                       const Geom &, int, int);

}  // namespace chan
