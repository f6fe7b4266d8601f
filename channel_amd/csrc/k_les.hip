// k_les.hip -- the learned subgrid-stress closure inside a coarse channel
// step, on the device (include/channel_closure.h): closure features of the
// resident field, the MLP, and the body force -div(tau) written straight
// into the context's static force, so that an LES step with the closure
// never leaves the GPU.  The reference has no subgrid model.
//
// Grid: rows iy = 0..ny of the dealiased physical grid Mx x Mz = 2nxd x nzd,
// x_j = j Lx / Mx, z_k = k Lz / Mz.  Spectral <-> physical transforms here
// are separable direct sums in FP32 (the LES grids are small: at 31x64x31 a
// transform of one row is 32 x 63 modes <-> 96 x 96 points); x and z
// derivatives are spectral, y derivatives the second-order differences of the
// stretched grid (one-sided three-point rows at the walls), applied to the
// spectral coefficients.
//
// Features of sample (iy, x, z), 46 values: the nine gradients du_c/dx_d
// (index 3c + d, d = x, y, z) at rows iy, iy-2, iy-1, iy+1, iy+2 (rows
// clamped to 0..ny), then y+ = min(y - ymin, ymax - y) u_tau / nu with u_tau
// from the mean wall shear of both walls (the wall-gradient stencils of
// outstats, dnsdata.f90:861-871).  Stresses: tau = (xx, yy, zz, xy, xz, yz).
#include <cmath>
#include <cstring>
#include <vector>

#include "../../include/channel_closure.h"
#include "ctx_internal.hpp"
#include "mlp_internal.hpp"

namespace chan {

struct LesState {
  int n = 0;                  // samples (ny+1) Mx Mz
  float *Gp = nullptr;        // [9][n] physical gradients
  float *Xf = nullptr;        // [n][46] features (host query)
  float *Y = nullptr;         // [n][6] MLP outputs
  float2 *T = nullptr;        // [6][ny+1][npair] spectral stresses
  float2 *twz = nullptr;      // [Mz] exp(+2 pi i k / Mz)
  float2 *phx = nullptr;      // [Nx][Mx up to XT] exp(+2 pi i ix xj / Mx)
  float2 *phxT = nullptr;     // [Mx][Nx up to XT] the same
  double *ydc = nullptr;      // [ny+1][3] y-difference coefficients of rows iy-1, iy, iy+1
  int *ydr = nullptr;         // [ny+1] first row of each stencil
  double *yplus = nullptr;    // [ny+1] wall distance in wall units
  float *norm = nullptr;      // [46 xmean][46 xscale][6 tmean][6 tscale][46 1/xscale]
  double *wall = nullptr;     // [2][5] wall-gradient stencils d140, d14n
};

void les_free(LesState *s) {
  if (!s) return;
  void *b[] = {s->Gp, s->Xf, s->Y, s->T, s->twz, s->phx, s->phxT, s->ydc, s->ydr, s->yplus, s->norm, s->wall};
  for (void *p : b)
    if (p) (void)hipFree(p);
  delete s;
}

namespace {

struct LesGeom {
  int nx, nz, ny, Nx, Nz, Ny, Mx, Mz, npair;
  size_t ps;
  double alfa0, beta0;
};

LesGeom les_geom(const chan_ctx *c) {
  LesGeom q;
  q.nx = c->g.nx;
  q.nz = c->g.nz;
  q.ny = c->g.ny;
  q.Nx = c->g.Nx;
  q.Nz = c->g.Nz;
  q.Ny = c->g.Ny;
  q.Mx = 2 * c->g.nxd;
  q.Mz = c->g.nzd;
  q.npair = c->g.npair;
  q.ps = c->g.ps;
  q.alfa0 = c->g.alfa0;
  q.beta0 = c->g.beta0;
  return q;
}

// a b with its fused operations written out, so that the sums formed from it do
// not depend on how the compiler would fuse them
__device__ __forceinline__ float2 cmulf(float2 a, float2 b) {
  return make_float2(fmaf(a.x, b.x, -(a.y * b.y)), fmaf(a.y, b.x, a.x * b.y));
}

// The transforms below are direct sums whose terms a thread adds in index order.
// One output per thread, they spent their time on a modulo and two or three LDS
// reads per term (943 us for the gradients at 31x64x31, 208 for the stresses);
// a thread now takes a tile of outputs that share each term's operand, with the
// phase index advanced by addition, and a block one derivative or stress of one
// row (65 and 66 us; the LDS reads of the shared operands bound them now).
constexpr int ZT = 8;     // x modes per thread in the z sums
constexpr int XT = 8;     // x points (or modes) per thread in the x sums
// threads: 8 x 96 points of the 96 x 96 grid in whole rounds (a force at 31x64x31 187 us,
// 219 with 256), and no slower on the others (48 x 48: 69 and 71, 24 x 24: 49.5 and 49.9)
constexpr int GT = 384;

__host__ __device__ __forceinline__ int round_up(int n, int k) { return (n + k - 1) / k * k; }
// The phases of the x sums, e^{+2 pi i ix xj / Mx}, come as [Nx][Mx up to XT] and
// transposed as [Mx][Nx up to XT].  k_les_grad stages them in LDS where they fit
// beside the rest (PL: 65 us for 74 at 31x64x31); k_les_tau, whose plane already
// fills LDS, reads them through the cache (66 us for 74: two blocks per CU
// instead of one).
inline size_t grad_phases(const LesGeom &q) { return sizeof(float2) * (size_t)q.Nx * round_up(q.Mx, XT); }
inline size_t tau_phases(const LesGeom &q) { return sizeof(float2) * (size_t)q.Mx * round_up(q.Nx, XT); }
// the rest of k_les_grad: S [Nz][Nx up to ZT], H [Nx][Mz], the z phases
inline size_t grad_lds(const LesGeom &q) {
  return sizeof(float2) * ((size_t)q.Nz * round_up(q.Nx, ZT) + (size_t)q.Nx * q.Mz + q.Mz);
}
constexpr size_t LDS_MAX = 160 * 1024;

// Derivative d = x, y, z of component c on row iy in physical space:
// Gp[3c + d][(iy Mx + x) Mz + z].  One block per (row, 3c + d).
template <bool PL>
__global__ __launch_bounds__(GT) void k_les_grad(const cx<double> *__restrict__ V, LesGeom q,
                                                 const double *__restrict__ ydc, const int *__restrict__ ydr,
                                                 const float2 *__restrict__ twz, const float2 *__restrict__ phx,
                                                 float *__restrict__ Gp) {
  extern __shared__ __align__(16) float2 sm[];
  const int NxP = round_up(q.Nx, ZT), MxP = round_up(q.Mx, XT);
  float2 *S = sm;                         // [Nz][NxP] spectral coefficients
  float2 *XL = S + (size_t)q.Nz * NxP;    // [Nx][MxP] phases of the x sum (PL)
  float2 *H = XL + (PL ? (size_t)q.Nx * MxP : 0);  // [Nx][Mz] after the z sum
  float2 *Z = H + (size_t)q.Nx * q.Mz;    // [Mz] e^{+2 pi i k / Mz}
  const int iy = blockIdx.x, c = blockIdx.y / 3, d = blockIdx.y % 3;
  const size_t cs = (size_t)c * q.Ny * q.ps;
  for (int i = threadIdx.x; i < q.Mz; i += GT) Z[i] = twz[i];
  if constexpr (PL)
    for (int i = threadIdx.x; i < q.Nx * MxP; i += GT) XL[i] = phx[i];
  for (int i = threadIdx.x; i < q.Nz * (NxP - q.Nx); i += GT)
    S[(i / (NxP - q.Nx)) * NxP + q.Nx + i % (NxP - q.Nx)] = make_float2(0.f, 0.f);
  for (int p = threadIdx.x; p < q.npair; p += GT) {
    const int ix = p / q.Nz, j = p % q.Nz, iz = j - q.nz;
    float2 s;
    if (d == 1) {
      const int r0 = ydr[iy];
      double re = 0.0, im = 0.0;
      for (int k = 0; k < 3; k++) {
        const cx<double> v = V[cs + (size_t)(r0 + k + 1) * q.ps + p];
        re += ydc[3 * iy + k] * v.x;
        im += ydc[3 * iy + k] * v.y;
      }
      s = make_float2((float)re, (float)im);
    } else {
      const cx<double> v = V[cs + (size_t)(iy + 1) * q.ps + p];
      const double k = d == 0 ? q.alfa0 * ix : q.beta0 * iz;  // i k v
      s = make_float2((float)(-k * v.y), (float)(k * v.x));
    }
    S[j * NxP + ix] = s;
  }
  __syncthreads();
  // z: H[ix][zk] = sum_iz S e^{+2 pi i iz zk / Mz}, ZT modes ix at a time
  for (int o = threadIdx.x; o < (NxP / ZT) * q.Mz; o += GT) {
    const int ix0 = (o / q.Mz) * ZT, zk = o % q.Mz;
    float2 acc[ZT];
#pragma unroll
    for (int k = 0; k < ZT; k++) acc[k] = make_float2(0.f, 0.f);
    int e = (int)(((long)(q.Mz - q.nz % q.Mz) * zk) % q.Mz);  // phase of iz = -nz
    for (int j = 0; j < q.Nz; j++) {
      const float2 w = Z[e];
      e += zk;
      e -= e >= q.Mz ? q.Mz : 0;
      const float2 *Sj = S + j * NxP + ix0;
#pragma unroll
      for (int k = 0; k < ZT; k++) {
        const float2 t = cmulf(Sj[k], w);
        acc[k].x += t.x;
        acc[k].y += t.y;
      }
    }
#pragma unroll
    for (int k = 0; k < ZT; k++)
      if (ix0 + k < q.Nx) H[(ix0 + k) * q.Mz + zk] = acc[k];
  }
  __syncthreads();
  // x: Hermitian sum over kx, XT points at a time
  float *G = Gp + (size_t)blockIdx.y * (q.ny + 1) * q.Mx * q.Mz + (size_t)iy * q.Mx * q.Mz;
  for (int o = threadIdx.x; o < (MxP / XT) * q.Mz; o += GT) {
    const int x0 = (o / q.Mz) * XT, zk = o % q.Mz;
    float g[XT];
#pragma unroll
    for (int k = 0; k < XT; k++) g[k] = 0.f;
    for (int ix = 1; ix < q.Nx; ix++) {
      const float2 h = H[ix * q.Mz + zk];
      const float2 *Xi = PL ? XL + ix * MxP + x0 : phx + (size_t)ix * MxP + x0;
#pragma unroll
      for (int k = 0; k < XT; k++) {
        const float2 t = cmulf(h, Xi[k]);
        g[k] += t.x;
      }
    }
    const float f0 = H[zk].x;
#pragma unroll
    for (int k = 0; k < XT; k++) {
      if (x0 + k >= q.Mx) break;
      float f = f0;
      f += 2.f * g[k];
      G[(size_t)(x0 + k) * q.Mz + zk] = f;
    }
  }
}

// u_tau from the mean wall shear of both walls, y+ of every row
__global__ void k_les_yplus(const cx<double> *__restrict__ V, LesGeom q, const double *__restrict__ wall,
                            const double *__restrict__ y, double ymin, double ymax, double ni,
                            double *__restrict__ yplus) {
  double db = 0.0, dt = 0.0;
  const int p0 = q.nz;  // pair (0, 0), component u
  for (int j = 0; j < 5; j++) {
    db += wall[j] * V[(size_t)j * q.ps + p0].x;                      // rows -1..3
    dt += wall[5 + j] * V[(size_t)(q.ny - 2 + j) * q.ps + p0].x;     // rows ny-3..ny+1
  }
  const double utau = sqrt(ni * 0.5 * (fabs(db) + fabs(dt)));
  for (int iy = threadIdx.x; iy <= q.ny; iy += blockDim.x) {
    const double yy = y[iy + 1];
    yplus[iy] = fmin(yy - ymin, ymax - yy) * utau / ni;
  }
}

// One thread per sample: its 46 features for the host query
__global__ __launch_bounds__(256) void k_les_features(const float *__restrict__ Gp, LesGeom q,
                                                      const double *__restrict__ yplus, float *__restrict__ Xf) {
  const int plane = q.Mx * q.Mz;
  const int n = (q.ny + 1) * plane;
  const int s = blockIdx.x * 256 + threadIdx.x;
  if (s >= n) return;
  const int iy = s / plane, o = s % plane;
  const int rows[5] = {iy, iy - 2, iy - 1, iy + 1, iy + 2};
#pragma unroll
  for (int k = 0; k < 5; k++) {
    const int r = min(max(rows[k], 0), q.ny);
#pragma unroll
    for (int j = 0; j < 9; j++) Xf[(size_t)s * 46 + 9 * k + j] = Gp[(size_t)j * n + (size_t)r * plane + o];
  }
  Xf[(size_t)s * 46 + 45] = (float)yplus[iy];
}

// LDS of k_les_tau: the plane [Mx][Mz], H [Mz][Nx up to ZT], the z phases
inline size_t tau_lds(const LesGeom &q) {
  return sizeof(float) * (size_t)round_up(q.Mx * q.Mz, 4) + sizeof(float2) * ((size_t)q.Mz * round_up(q.Nx, ZT) + q.Mz);
}

// Spectral stresses of row iy, component qq: T = (1/(Mx Mz)) sum tau e^{-i(kx x + kz z)}
__global__ __launch_bounds__(GT) void k_les_tau(const float *__restrict__ Y, LesGeom q, const float *__restrict__ norm,
                                                const float2 *__restrict__ twz, const float2 *__restrict__ phxT,
                                                float2 *__restrict__ T) {
  extern __shared__ __align__(16) float2 sm[];
  const int NxP = round_up(q.Nx, XT);
  static_assert(XT == ZT, "one padding of the x modes");
  float *P = reinterpret_cast<float *>(sm);                                // [Mx][Mz]
  float2 *H = reinterpret_cast<float2 *>(P + round_up(q.Mx * q.Mz, 4));    // [Mz][NxP]
  float2 *Z = H + (size_t)q.Mz * NxP;                                      // [Mz]
  const int iy = blockIdx.x, qq = blockIdx.y;
  const int plane = q.Mx * q.Mz;
  const float tm = norm[92 + qq], ts = norm[98 + qq];
  for (int i = threadIdx.x; i < q.Mz; i += GT) Z[i] = twz[i];
  for (int o = threadIdx.x; o < plane; o += GT) P[o] = Y[((size_t)iy * plane + o) * 6 + qq] * ts + tm;
  __syncthreads();
  for (int o = threadIdx.x; o < (NxP / XT) * q.Mz; o += GT) {
    const int ix0 = (o / q.Mz) * XT, zk = o % q.Mz;
    float2 acc[XT];
#pragma unroll
    for (int k = 0; k < XT; k++) acc[k] = make_float2(0.f, 0.f);
    for (int xj = 0; xj < q.Mx; xj++) {
      const float v = P[xj * q.Mz + zk];
      const float2 *w = phxT + (size_t)xj * NxP + ix0;
#pragma unroll
      for (int k = 0; k < XT; k++) {
        acc[k].x = fmaf(v, w[k].x, acc[k].x);
        acc[k].y = fmaf(-v, w[k].y, acc[k].y);  // conj
      }
    }
#pragma unroll
    for (int k = 0; k < XT; k++) H[zk * NxP + ix0 + k] = make_float2(acc[k].x / q.Mx, acc[k].y / q.Mx);
  }
  __syncthreads();
  for (int o = threadIdx.x; o < (NxP / ZT) * q.Nz; o += GT) {
    const int ix0 = (o / q.Nz) * ZT, j = o % q.Nz, iz = j - q.nz;
    float2 acc[ZT];
#pragma unroll
    for (int k = 0; k < ZT; k++) acc[k] = make_float2(0.f, 0.f);
    const int de = ((iz % q.Mz) + q.Mz) % q.Mz;  // phase step of iz
    int e = 0;
    for (int zk = 0; zk < q.Mz; zk++) {
      const float2 w = make_float2(Z[e].x, -Z[e].y);
      e += de;
      e -= e >= q.Mz ? q.Mz : 0;
#pragma unroll
      for (int k = 0; k < ZT; k++) {
        const float2 t = cmulf(H[zk * NxP + ix0 + k], w);
        acc[k].x += t.x;
        acc[k].y += t.y;
      }
    }
#pragma unroll
    for (int k = 0; k < ZT; k++)
      if (ix0 + k < q.Nx)
        T[((size_t)qq * (q.ny + 1) + iy) * q.npair + (ix0 + k) * q.Nz + j] =
            make_float2(acc[k].x / q.Mz, acc[k].y / q.Mz);
  }
}

// F_i = -(d_x tau_xi + d_y tau_yi + d_z tau_zi) on rows 0..ny; ghost rows 0
__global__ __launch_bounds__(256) void k_les_div(const float2 *__restrict__ T, LesGeom q,
                                                 const double *__restrict__ ydc, const int *__restrict__ ydr,
                                                 cx<double> *__restrict__ F) {
  const int p = blockIdx.x * 256 + threadIdx.x, row = blockIdx.y;  // device row: iy + 1
  if (p >= q.npair) return;
  const int ix = p / q.Nz, iz = p % q.Nz - q.nz;
  const double kx = q.alfa0 * ix, kz = q.beta0 * iz;
  const size_t cs = (size_t)q.Ny * q.ps;
  if (row == 0 || row == q.ny + 2) {
    for (int i = 0; i < 3; i++) F[i * cs + (size_t)row * q.ps + p] = cx<double>{0.0, 0.0};
    return;
  }
  const int iy = row - 1;
  auto Tq = [&](int qq, int r) {
    const float2 t = T[((size_t)qq * (q.ny + 1) + r) * q.npair + p];
    return cx<double>{(double)t.x, (double)t.y};
  };
  auto dyq = [&](int qq) {
    const int r0 = ydr[iy];
    cx<double> a{0.0, 0.0};
    for (int k = 0; k < 3; k++) {
      const cx<double> t = Tq(qq, r0 + k);
      a.x += ydc[3 * iy + k] * t.x;
      a.y += ydc[3 * iy + k] * t.y;
    }
    return a;
  };
  // (x-stress, y-stress, z-stress) of each momentum component i
  const int qx[3] = {0, 3, 4}, qy[3] = {3, 1, 5}, qz[3] = {4, 5, 2};
  for (int i = 0; i < 3; i++) {
    const cx<double> a = Tq(qx[i], iy), b = dyq(qy[i]), cz = Tq(qz[i], iy);
    // i kx a + b + i kz c
    const double re = -kx * a.y + b.x - kz * cz.y, im = kx * a.x + b.y + kz * cz.x;
    F[i * cs + (size_t)row * q.ps + p] = cx<double>{-re, -im};
  }
}

template <class T>
int lmal(T **p, size_t n) {
  hipError_t e = hipMalloc((void **)p, n * sizeof(T) + 256);
  if (e != hipSuccess) return set_error((int)e, "hipMalloc of %zu bytes failed", n * sizeof(T));
  return 0;
}

#define LCHK(expr)                                                                           \
  do {                                                                                       \
    hipError_t e_ = (expr);                                                                  \
    if (e_ != hipSuccess) return set_error((int)e_, "%s: %s", #expr, hipGetErrorString(e_)); \
  } while (0)

// the closure buffers of c, made on the first call
int les_state(chan_ctx *c, LesState **out) {
  if (c->les) {
    *out = c->les;
    return 0;
  }
  const LesGeom q = les_geom(c);
  LesState *s = new LesState();
  s->n = (q.ny + 1) * q.Mx * q.Mz;
  int rc;
  auto bail = [&](int code) {
    les_free(s);
    return code;
  };
  const size_t n = (size_t)s->n;
  if ((rc = lmal(&s->Gp, n * 9)) || (rc = lmal(&s->Y, n * 6)) || (rc = lmal(&s->T, (size_t)6 * (q.ny + 1) * q.npair)) ||
      (rc = lmal(&s->twz, (size_t)q.Mz)) || (rc = lmal(&s->phx, grad_phases(q) / sizeof(float2))) || (rc = lmal(&s->phxT, tau_phases(q) / sizeof(float2))) ||
      (rc = lmal(&s->ydc, (size_t)3 * (q.ny + 1))) || (rc = lmal(&s->ydr, (size_t)q.ny + 1)) ||
      (rc = lmal(&s->yplus, (size_t)q.ny + 1)) || (rc = lmal(&s->norm, (size_t)mlp::NORM_RECIP + 46)) || (rc = lmal(&s->wall, (size_t)10)))
    return bail(rc);
  // twiddles
  std::vector<float2> tz(q.Mz), tx(q.Mx);
  const double pi2 = 2.0 * 3.14159265358979323846;
  for (int k = 0; k < q.Mz; k++) tz[k] = make_float2((float)cos(pi2 * k / q.Mz), (float)sin(pi2 * k / q.Mz));
  for (int k = 0; k < q.Mx; k++) tx[k] = make_float2((float)cos(pi2 * k / q.Mx), (float)sin(pi2 * k / q.Mx));
  const int MxP = round_up(q.Mx, XT), NxP = round_up(q.Nx, XT);
  std::vector<float2> px((size_t)q.Nx * MxP), pxT((size_t)q.Mx * NxP);
  for (int ix = 0; ix < q.Nx; ix++)
    for (int xj = 0; xj < MxP; xj++) px[(size_t)ix * MxP + xj] = tx[(int)((long long)ix * xj % q.Mx)];
  for (int xj = 0; xj < q.Mx; xj++)
    for (int ix = 0; ix < NxP; ix++) pxT[(size_t)xj * NxP + ix] = tx[(int)((long long)ix * xj % q.Mx)];
  // second-order differences on the stretched rows 0..ny (numpy.gradient, edge_order 2)
  const double *y = c->hs.y + 1;  // y[iy], iy = 0..ny
  const int ny = q.ny;
  std::vector<double> dc(3 * (ny + 1));
  std::vector<int> dr(ny + 1);
  for (int i = 0; i <= ny; i++) {
    double *w = &dc[3 * i];
    if (i == 0) {
      const double h1 = y[1] - y[0], h2 = y[2] - y[1];
      w[0] = -(2 * h1 + h2) / (h1 * (h1 + h2));
      w[1] = (h1 + h2) / (h1 * h2);
      w[2] = -h1 / (h2 * (h1 + h2));
      dr[i] = 0;
    } else if (i == ny) {
      const double h1 = y[ny - 1] - y[ny - 2], h2 = y[ny] - y[ny - 1];
      w[0] = h2 / (h1 * (h1 + h2));
      w[1] = -(h1 + h2) / (h1 * h2);
      w[2] = (2 * h2 + h1) / (h2 * (h1 + h2));
      dr[i] = ny - 2;
    } else {
      const double h1 = y[i] - y[i - 1], h2 = y[i + 1] - y[i];
      w[0] = -h2 / (h1 * (h1 + h2));
      w[1] = (h2 - h1) / (h1 * h2);
      w[2] = h1 / (h2 * (h1 + h2));
      dr[i] = i - 1;
    }
  }
  double wall[10];
  std::memcpy(wall, c->hs.bnd[B_D140], 5 * sizeof(double));
  std::memcpy(wall + 5, c->hs.bnd[B_D14N], 5 * sizeof(double));
  if (hipMemcpy(s->twz, tz.data(), tz.size() * sizeof(float2), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(s->phx, px.data(), px.size() * sizeof(float2), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(s->phxT, pxT.data(), pxT.size() * sizeof(float2), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(s->ydc, dc.data(), dc.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(s->ydr, dr.data(), dr.size() * sizeof(int), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(s->wall, wall, sizeof wall, hipMemcpyHostToDevice) != hipSuccess)
    return bail(set_error(CHAN_E_STATE, "upload of the closure set-up failed"));
  c->les = s;
  *out = s;
  return 0;
}

// The closure runs where one row's transform fits in 64 KiB: spectral
// coefficients and one z-transformed row, or one physical plane and the same.
int les_fits(const LesGeom &q, bool stresses) {
  const size_t h = sizeof(float2) * (size_t)q.Nx * q.Mz;
  const size_t b = h + (stresses ? sizeof(float) * ((size_t)q.Mx * q.Mz + 1) + 16 : sizeof(float2) * (size_t)q.npair);
  if (b > 64 * 1024) return set_error(CHAN_E_SIZE, "closure grid too large (%zu bytes of LDS per row)", b);
  return 0;  // grad_lds and tau_lds, at most twice that for the padding of Nx >= 4, then fit in 160 KiB
}

// gradients and y+ of the resident field
int les_gradients(chan_ctx *c, LesState *s) {
  const LesGeom q = les_geom(c);
  int rc;
  if ((rc = les_fits(q, false))) return rc;
  const size_t lds = grad_lds(q), all = lds + grad_phases(q);
  if (all <= LDS_MAX)
    hipLaunchKernelGGL(k_les_grad<true>, dim3(q.ny + 1, 9), dim3(GT), all, c->st, c->V, q, s->ydc, s->ydr, s->twz, s->phx,
                       s->Gp);
  else
    hipLaunchKernelGGL(k_les_grad<false>, dim3(q.ny + 1, 9), dim3(GT), lds, c->st, c->V, q, s->ydc, s->ydr, s->twz,
                       s->phx, s->Gp);
  LCHK(hipGetLastError());
  hipLaunchKernelGGL(k_les_yplus, dim3(1), dim3(256), 0, c->st, c->V, q, s->wall, c->y, c->prm.ymin, c->prm.ymax,
                     c->prm.ni, s->yplus);
  LCHK(hipGetLastError());
  return 0;
}

// the closure's force on the resident field into F0, enqueued on the context's stream
int les_force(chan_ctx *c, LesState *s, chan_mlp *m, const float *norm, size_t norm_bytes, bool quick) {
  int rc;
  LCHK(hipMemcpyAsync(s->norm, norm, norm_bytes, hipMemcpyHostToDevice, c->st));
  if ((rc = les_gradients(c, s))) return rc;
  const LesGeom q = les_geom(c);
  LCHK(mlp::forward_gradients(m, mlp::LesSource{s->Gp, s->norm, s->yplus, s->n, q.Mx * q.Mz, q.ny, quick}, s->Y, c->st));
  if ((rc = les_fits(q, true))) return rc;
  hipLaunchKernelGGL(k_les_tau, dim3(q.ny + 1, 6), dim3(GT), tau_lds(q), c->st, s->Y, q, s->norm, s->twz, s->phxT, s->T);
  LCHK(hipGetLastError());
  if (!c->F0) {
    if ((rc = lmal(&c->F0, 3 * (size_t)q.Ny * q.ps))) return rc;
    LCHK(hipMemsetAsync(c->F0, 0, sizeof(cx<double>) * 3 * (size_t)q.Ny * q.ps, c->st));
  }
  hipLaunchKernelGGL(k_les_div, dim3((q.npair + 255) / 256, q.Ny), dim3(256), 0, c->st, s->T, q, s->ydc, s->ydr, c->F0);
  LCHK(hipGetLastError());
  return 0;
}

}  // namespace
}  // namespace chan

using namespace chan;

extern "C" {

int chan_les_features(chan_ctx *c, float *X) {
  if (!c || !X) return set_error(CHAN_E_ARG, "null argument");
  if (!c->field_set) return set_error(CHAN_E_STATE, "closure features before set_field");
  LesState *s;
  int rc;
  if ((rc = les_state(c, &s))) return rc;
  if (!s->Xf && (rc = lmal(&s->Xf, (size_t)s->n * 46))) return rc;
  if ((rc = les_gradients(c, s))) return rc;
  hipLaunchKernelGGL(k_les_features, dim3((s->n + 255) / 256), dim3(256), 0, c->st, s->Gp, les_geom(c), s->yplus, s->Xf);
  LCHK(hipGetLastError());
  LCHK(copy_to_host(c->stage, X, s->Xf, sizeof(float) * 46 * (size_t)s->n, c->st));
  return 0;
}

int chan_les_samples(const chan_ctx *c, int64_t *n) {
  if (!c || !n) return set_error(CHAN_E_ARG, "null argument");
  *n = (int64_t)(c->g.ny + 1) * 2 * c->g.nxd * c->g.nzd;
  return 0;
}

int chan_les_closure_force(chan_ctx *c, chan_mlp *m, const float *norm) {
  if (!c || !m || !norm) return set_error(CHAN_E_ARG, "null argument");
  if (!c->field_set) return set_error(CHAN_E_STATE, "closure force before set_field");
  LesState *s;
  int rc;
  if ((rc = les_state(c, &s))) return rc;
  for (int j = 0; j < 46; j++)
    if (!(norm[46 + j] > 0.0f)) return set_error(CHAN_E_ARG, "feature scale %d is not positive", j);
  float nv[mlp::NORM_RECIP + 46];
  bool quick = true;
  std::memcpy(nv, norm, sizeof(float) * mlp::NORM_RECIP);
  for (int j = 0; j < 46; j++) {
    nv[mlp::NORM_RECIP + j] = 1.0f / norm[46 + j];
    quick = quick && norm[46 + j] >= 1.0f / mlp::SPAN_D && norm[46 + j] <= mlp::SPAN_D;
  }
  rc = les_force(c, s, m, nv, sizeof nv, quick);
  const hipError_t end = hipStreamSynchronize(c->st);  // until then nv may still be read
  if (rc) return rc;
  LCHK(end);
  return 0;
}

}  // extern "C"
