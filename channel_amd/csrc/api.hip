// api.hip -- the C-ABI of include/channel_hip.h: device-resident state of
// one channel DNS, set-up, field exchange in the reference layout and the
// launch sequences of buildrhs / linsolve / the RK3 time loop.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <algorithm>
#include <cstddef>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "../../include/channel_hip.h"
#include "chan_internal.hpp"
#include "ctx_internal.hpp"

using namespace chan;

namespace {

thread_local char g_err[1024] = "";

int fail(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof g_err, fmt, ap);
  va_end(ap);
  return code;
}

}  // namespace

// error reporting shared with the closure library part (k_mlp.hip)
int chan::set_error(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof g_err, fmt, ap);
  va_end(ap);
  return code;
}

namespace {

#define HIPCHK(expr)                                                                              \
  do {                                                                                            \
    hipError_t e_ = (expr);                                                                       \
    if (e_ != hipSuccess) return fail((int)e_, "%s: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__); \
  } while (0)

// RK3 coefficients of Rai & Moin (dnsdata.f90:70-72)
const double RK1[3] = {120.0 / 32.0, 2.0, 0.0};
const double RK2[3] = {120.0 / 8.0, 50.0 / 8.0, 34.0 / 8.0};
const double RK3[3] = {120.0 / 20.0, 90.0 / 20.0, 50.0 / 20.0};

// ---------------------------------------------------- layout transposes --
// host layout: [c][pair][row] (the reference's V(iy,iz,ix,c), iy fastest);
// device layout: [c][row][pair] with plane stride ps.
constexpr int TT = 32;
__global__ __launch_bounds__(TT * 8) void k_to_dev(const cx<double> *__restrict__ in, cx<double> *__restrict__ out, Geom g) {
  __shared__ cx<double> tile[TT][TT + 1];
  const int c = blockIdx.z;
  const int p0 = blockIdx.x * TT, r0 = blockIdx.y * TT;
  const cx<double> *src = in + (size_t)c * g.npair * g.Ny;
  cx<double> *dst = out + (size_t)c * g.Ny * g.ps;
  for (int k = threadIdx.y; k < TT; k += 8) {
    const int p = p0 + k, r = r0 + threadIdx.x;
    if (p < g.npair && r < g.Ny) tile[k][threadIdx.x] = src[(size_t)p * g.Ny + r];
  }
  __syncthreads();
  for (int k = threadIdx.y; k < TT; k += 8) {
    const int r = r0 + k, p = p0 + threadIdx.x;
    if (p < g.npair && r < g.Ny) dst[(size_t)r * g.ps + p] = tile[threadIdx.x][k];
  }
}
__global__ __launch_bounds__(TT * 8) void k_to_host(const cx<double> *__restrict__ in, cx<double> *__restrict__ out, Geom g) {
  __shared__ cx<double> tile[TT][TT + 1];
  const int c = blockIdx.z;
  const int p0 = blockIdx.x * TT, r0 = blockIdx.y * TT;
  const cx<double> *src = in + (size_t)c * g.Ny * g.ps;
  cx<double> *dst = out + (size_t)c * g.npair * g.Ny;
  for (int k = threadIdx.y; k < TT; k += 8) {
    const int r = r0 + k, p = p0 + threadIdx.x;
    if (p < g.npair && r < g.Ny) tile[k][threadIdx.x] = src[(size_t)r * g.ps + p];
  }
  __syncthreads();
  for (int k = threadIdx.y; k < TT; k += 8) {
    const int p = p0 + k, r = r0 + threadIdx.x;
    if (p < g.npair && r < g.Ny) dst[(size_t)p * g.Ny + r] = tile[threadIdx.x][k];
  }
}

// What outstats reads on the host: five rows of u's and w's (0,0) columns at each
// wall and the device scalars.  Pinned memory that the kernel writes itself, so
// that a step ends with one launch and a wait: a copy engine's transfer to
// pageable memory took 20 us more, of 250 for a step of a 15x32x15 field.
struct StepRow {
  double lo[2][5], hi[2][5];
  DevScalars sc;
};
// The scalars and the running maxima as they lie on the device, for the host: one copy
// brings both (a kernel that folded them first made chan_get_scalars 3 to 10 us longer).
struct ScalarBlock {
  DevScalars sc;
  alignas(128) unsigned long long cfl[CFL_SLOTS * CFL_STRIDE];
};
// The largest of the CFL_SLOTS running maxima and before, which start again at 0;
// called by one whole wave.
__device__ __forceinline__ unsigned long long take_cfl(unsigned long long *slots, unsigned long long before) {
  static_assert(CFL_SLOTS == 64, "a slot per lane");
  unsigned long long *mine = slots + threadIdx.x * CFL_STRIDE, m = *mine;
  *mine = 0ull;
  m = m > before ? m : before;
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) {
    const unsigned long long o = __shfl_xor(m, s, 64);
    m = o > m ? o : m;
  }
  return m;
}
// The running CFL maximum restarts at 0.
__global__ void k_step_row(const cx<double> *__restrict__ V, StepRow *__restrict__ out, DevScalars *sc,
                           unsigned long long *cfl_max, Geom g) {
  const int t = threadIdx.x;
  DevScalars s = *sc;
  s.cfl_bits = take_cfl(cfl_max, s.cfl_bits);
  if (t == 0) {
    out->sc = s;
    sc->cfl_bits = 0ull;
  }
  if (t >= 20) return;
  const int comp = t / 5 % 2, j = t % 5, r = t < 10 ? j : g.Ny - 5 + j;
  (t < 10 ? out->lo : out->hi)[comp][j] = V[((size_t)2 * comp * g.Ny + r) * g.ps + g.nz].x;
}

// grid-stride streaming copy of n 32-byte elements
__global__ __launch_bounds__(256) void k_copy(const double4 *__restrict__ a, double4 *__restrict__ b, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) b[i] = a[i];
}

// the table of k_solve_lds (SROW)
void solve_table(const HostSetup &h, int ny, std::vector<double> &t) {
  const int n = ny - 1, m = n / 2;
  t.assign((size_t)n * SROW, 0.0);
  const int src[4] = {0, 10, 15, 5};  // d0, d2, d4, d1
  for (int r = 0; r < n; r++)
    for (int k = 0; k < 4; k++)
      for (int j = 0; j < 5; j++) t[(size_t)r * SROW + 5 * k + j] = h.der[(size_t)r * 20 + src[k] + (r < m ? 4 - j : j)];
  // D0 factors: from the upper wall the set-up's, from the lower one the same
  // elimination in the mirrored rows
  for (int r = n - 1; r >= m; r--)
    for (int j = 0; j < 5; j++) t[(size_t)r * SROW + 20 + j] = h.d0fac[(size_t)r * 5 + j];
  double l1[2] = {0, 0}, l2[2] = {0, 0};
  for (int r = 0; r < m; r++) {
    double *A = &t[(size_t)r * SROW + 20];
    for (int j = 0; j < 5; j++) A[j] = t[(size_t)r * SROW + j];
    if (r == 0) A[3] = A[4] = 0.0;  // the wall columns
    if (r == 1) A[4] = 0.0;
    A[3] -= A[4] * l2[1];
    A[2] -= A[4] * l2[0];
    A[2] -= A[3] * l1[1];
    A[1] -= A[3] * l1[0];
    A[2] = 1.0 / A[2];
    A[0] *= A[2];
    A[1] *= A[2];
    for (int j = 0; j < 2; j++) {
      l2[j] = l1[j];
      l1[j] = A[j];
    }
  }
}

template <typename T>
void twiddles(std::vector<cx<T>> &w, int n) {
  w.resize((size_t)fft::tw_table_size(n));
  fft::build_twiddles(w.data(), n);
}
// the x pass's table: 768-point rows use the four-step transform, 1536-point
// rows its two-wave form
template <typename T>
void twiddles_x(std::vector<cx<T>> &w, int n) {
  if (n == 1536) {
    w.resize((size_t)fft::FS2_TW);
    fft::build_fs1536_twiddles(w.data());
    return;
  }
  if (n != 768) return twiddles(w, n);
  w.resize((size_t)fft::FS_TW);
  fft::build_fs768_twiddles(w.data());
}

}  // namespace

namespace chan {
hipError_t launch_to_device_layout(hipStream_t st, const cx<double> *in, cx<double> *out, const Geom &g) {
  dim3 grid((unsigned)((g.npair + TT - 1) / TT), (unsigned)((g.Ny + TT - 1) / TT), 3);
  hipLaunchKernelGGL(k_to_dev, grid, dim3(TT, 8), 0, st, in, out, g);
  return hipGetLastError();
}
hipError_t launch_to_host_layout(hipStream_t st, const cx<double> *in, cx<double> *out, const Geom &g) {
  dim3 grid((unsigned)((g.npair + TT - 1) / TT), (unsigned)((g.Ny + TT - 1) / TT), 3);
  hipLaunchKernelGGL(k_to_host, grid, dim3(TT, 8), 0, st, in, out, g);
  return hipGetLastError();
}
}  // namespace chan

namespace {

int kid(chan_ctx *c, const char *name) {
  for (size_t i = 0; i < c->names.size(); i++)
    if (c->names[i] == name) return (int)i;
  c->names.push_back(name);
  c->counts.push_back(0);
  c->ms.push_back(0.0);
  return (int)c->names.size() - 1;
}

hipEvent_t get_event(chan_ctx *c) {
  if (!c->pool.empty()) {
    hipEvent_t e = c->pool.back();
    c->pool.pop_back();
    return e;
  }
  hipEvent_t e;
  if (hipEventCreate(&e) != hipSuccess) return nullptr;
  return e;
}

int harvest(chan_ctx *c) {
  for (auto &r : c->pend) {
    HIPCHK(hipEventSynchronize(r.b));
    float t = 0;
    HIPCHK(hipEventElapsedTime(&t, r.a, r.b));
    c->counts[r.id] += 1;
    c->ms[r.id] += t;
    c->pool.push_back(r.a);
    c->pool.push_back(r.b);
  }
  c->pend.clear();
  return 0;
}

// runs `launch` on the context's stream, bracketed by events when timing
template <class F>
int timed(chan_ctx *c, const char *name, F launch) {
  hipEvent_t a = nullptr, b = nullptr;
  if (c->timing) {
    if (c->pend.size() > 8192) {
      int rc = harvest(c);
      if (rc) return rc;
    }
    a = get_event(c);
    b = get_event(c);
    if (!a || !b) return fail(CHAN_E_STATE, "hipEventCreate failed");
    HIPCHK(hipEventRecord(a, c->st));
  }
  hipError_t e = launch();
  if (e != hipSuccess) return fail((int)e, "launch of %s failed: %s", name, hipGetErrorString(e));
  if (c->timing) {
    HIPCHK(hipEventRecord(b, c->st));
    c->pend.push_back({kid(c, name), a, b});
  }
  return 0;
}

int dalloc_bytes(void **p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes + 256);
  if (e != hipSuccess) return fail((int)e, "hipMalloc of %zu bytes failed: %s", bytes, hipGetErrorString(e));
  return 0;
}

template <class T>
int dalloc(T **p, size_t n) {
  hipError_t e = hipMalloc((void **)p, n * sizeof(T) + 256);
  if (e != hipSuccess) return fail((int)e, "hipMalloc of %zu bytes failed: %s", n * sizeof(T), hipGetErrorString(e));
  return 0;
}

// A context's small device arrays in one allocation, brought there by one copy: with
// one of each per array, chan_create took 95 us longer at 15x32x15 and 310 at 95x128x95.
struct Tables {
  std::vector<char> image;
  std::vector<std::pair<void **, size_t>> wanted;  // whom to tell where an array came to lie
  template <class T>
  size_t add(const T *src, size_t n) {
    const size_t at = image.size();
    image.resize((at + n * sizeof(T) + 255) / 256 * 256);
    std::memcpy(image.data() + at, src, n * sizeof(T));
    return at;
  }
  template <class T>
  size_t add(const std::vector<T> &v) {
    return add(v.data(), v.size());
  }
  template <class T>
  void want(T **p, size_t at) {
    wanted.push_back({(void **)p, at});
  }
  void place(char *base) {
    for (auto &w : wanted) *w.first = base + w.second;
  }
};

ForceArgs force_args(const chan_ctx *c) {
  ForceArgs a;
  a.V = c->V;
  a.F0 = c->F0;
  a.gain = c->gain;
  a.der = c->der;
  a.derF = c->derF;
  for (int k = 0; k < 3; k++) a.src[k] = c->gain ? c->src[k] : -1;
  a.out = nullptr;
  a.g = c->g;
  return a;
}

double cfl_value(const DevScalars &s) {
  double v;
  std::memcpy(&v, &s.cfl_bits, sizeof v);
  return v;
}

}  // namespace

extern "C" {

int chan_abi_version(void) { return CHAN_ABI_VERSION; }
const char *chan_last_error(void) { return g_err; }

int chan_create(const chan_params *p, chan_ctx **out) {
  if (!p || !out) return fail(CHAN_E_ARG, "null argument");
  *out = nullptr;
  if (p->nx < 1 || p->nz < 1 || p->ny < 8) return fail(CHAN_E_ARG, "need nx >= 1, nz >= 1, ny >= 8 (got %d %d %d)", p->nx, p->ny, p->nz);
  if (p->precision != CHAN_FP64 && p->precision != CHAN_SPLIT)
    return fail(CHAN_E_ARG, "precision mode %d is not available", p->precision);
  if (p->cpi && p->cpi_type != 0 && p->cpi_type != 1) return fail(CHAN_E_CPITYPE, "Wrong selection of CPI_Type (%d)", p->cpi_type);
  if (!(p->alfa0 > 0) || !(p->beta0 > 0) || !(p->ni > 0) || !(p->ymax > p->ymin) || !(p->a > 0))
    return fail(CHAN_E_ARG, "alfa0, beta0, ni, a must be positive and ymax > ymin");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(CHAN_E_NODEV, "no HIP device");
  chan_ctx *c = new chan_ctx();
  c->prm = *p;
  c->split = p->precision == CHAN_SPLIT;
  setup_build(c->hs, p->nx, p->ny, p->nz, p->alfa0, p->beta0, p->a, p->ymin, p->ymax);
  const HostSetup &h = c->hs;
  // the x pass holds at most (E+2)/3 x modes per thread, i.e. Nx <= 2nxd/3,
  // which fftFIT's nxd >= 3(nx+1)/2 guarantees
  if (!fft_size_supported(h.nzd) || !fft_size_supported(2 * h.nxd) || h.nzd % ZB != 0 || 3 * (p->nx + 1) > 2 * h.nxd) {
    int rc;
    if (3 * (p->nx + 1) > 2 * h.nxd)
      rc = fail(CHAN_E_SIZE,
                "nx=%d: the x pass needs 3(nx+1) <= 2nxd, but fftFIT keeps nxd=%d (3(nx+1)/2 rounded down is "
                "already 2^k or 3*2^k), so 3(nx+1)=%d > 2nxd=%d; choose another nx (nx=%d or %d)",
                p->nx, h.nxd, 3 * (p->nx + 1), 2 * h.nxd, p->nx - 1, p->nx + 1);
    else
      rc = fail(CHAN_E_SIZE, "transform sizes nzd=%d, 2nxd=%d are not supported", h.nzd, 2 * h.nxd);
    setup_free(c->hs);
    delete c;
    return rc;
  }
  Geom &g = c->g;
  g.nx = p->nx;
  g.ny = p->ny;
  g.nz = p->nz;
  g.Nx = p->nx + 1;
  g.Nz = 2 * p->nz + 1;
  g.Ny = p->ny + 3;
  g.nxd = h.nxd;
  g.nzd = h.nzd;
  g.npair = g.Nx * g.Nz;
  g.ps = ((size_t)g.npair + 1 + 63) / 64 * 64;  // one spare slot: the ucor solve
  g.alfa0 = p->alfa0;
  g.beta0 = p->beta0;
  {
    int dev = 0, ncu = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || ncu < 1)
      ncu = 256;
    g.ncu = ncu;
  }
  c->time = p->time;
  c->deltat = p->deltat;

  int rc = 0;
  auto bail = [&](int code) {
    chan_destroy(c);
    return code;
  };
  if (hipStreamCreate(&c->st) != hipSuccess) return bail(fail(CHAN_E_STATE, "hipStreamCreate failed"));
  const size_t plane = g.ps, NyP = (size_t)g.Ny * plane;
  const size_t slab = (size_t)g.nzd * g.Nx;  // one component of one plane in physical z
  if ((rc = dalloc(&c->V, 3 * NyP))) return bail(rc);
  if ((rc = dalloc(&c->rhs, 2 * (size_t)(g.ny - 1) * plane))) return bail(rc);
  const size_t factors = solve_factors(g);
  if (factors && (rc = dalloc(&c->L, factors))) return bail(rc);
  if (hipHostMalloc(&c->step_row, sizeof(StepRow), hipHostMallocDefault) != hipSuccess)
    return bail(fail(CHAN_E_STATE, "hipHostMalloc failed"));
  const size_t esz = c->split ? sizeof(cx<float>) : sizeof(cx<double>);
  if ((rc = dalloc_bytes(&c->old, 2 * (size_t)(g.ny - 1) * plane * esz))) return bail(rc);
  // B doubles as the staging area of the field and rhs transposes, which
  // needs 3*Ny*npair complex FP64 <= NPROD*Ny*slab*esz (nzd >= 3 nz), P as the
  // device layout of a force, 3*Ny*ps complex FP64
  if ((rc = dalloc_bytes(&c->A, 3 * (size_t)g.Ny * slab * esz))) return bail(rc);
  if ((rc = dalloc_bytes(&c->B, NPROD * (size_t)g.Ny * slab * esz))) return bail(rc);
  if ((rc = dalloc_bytes(&c->P, NyP * (NPROD * esz > 48 ? NPROD * esz : 48)))) return bail(rc);
  // no mode that is kept may alias: more than 3 nz points in z; 3 (nx + 1) in x,
  // which the x pass's slots need
  c->nzs = alias_free_z(3 * g.nz + 1, g.nzd);
  c->mxs = alias_free_x(3 * g.Nx, 2 * g.nxd, (unsigned)(c->nzs / ZB * g.Ny), g.ncu, c->split);
  Tables tb;
  auto twiddle_tables = [&](auto proto) {
    typedef decltype(proto) W;
    std::vector<W> tw;
    auto z = [&](int n) {
      twiddles(tw, n);
      return tb.add(tw);
    };
    auto x = [&](int n) {
      twiddles_x(tw, n);
      return tb.add(tw);
    };
    const size_t tz = z(g.nzd), tx = x(2 * g.nxd);
    const size_t tzs = c->nzs == g.nzd ? tz : z(c->nzs);
    const size_t txs = c->mxs == 2 * g.nxd ? tx : (c->mxs == c->nzs ? tzs : x(c->mxs));  // 9*2^k: one table
    tb.want(&c->twz, tz);
    tb.want(&c->twx, tx);
    tb.want(&c->twzs, tzs);
    tb.want(&c->twxs, txs);
  };
  if (c->split)
    twiddle_tables(cx<float>{});
  else
    twiddle_tables(cx<double>{});
  tb.want(&c->der, tb.add(h.der, (size_t)20 * (g.ny - 1)));
  tb.want(&c->d0fac, tb.add(h.d0fac, (size_t)5 * (g.ny + 1)));
  tb.want(&c->y, tb.add(h.y, (size_t)g.Ny));
  tb.want(&c->dy, tb.add(h.dy, (size_t)g.ny + 1));
  {
    // row r's weights in the stencils of the interior rows r-2..r+2; those of
    // a body force have its wall rows folded in: F(0) = F(ny) = 0, and the
    // ghost values F(-1) = -(d4[2] F(1) + d4[3] F(2) + d4[4] F(3)) / d4[0] of
    // row 1 and F(ny+1) of row ny-1 likewise
    std::vector<double> t((size_t)g.Ny * 20, 0.0), tf((size_t)g.Ny * 10, 0.0);
    for (int r = -1; r <= g.ny + 1; r++)
      for (int m = 0; m < 5; m++) {
        const int iy = r - 2 + m, j = 4 - m;
        if (iy < 1 || iy > g.ny - 1) continue;
        const double *d = h.der + (size_t)(iy - 1) * 20, *d4 = d + 15;
        for (int f = 0; f < 4; f++) t[(size_t)(r + 1) * 20 + 4 * m + f] = d[5 * f + j];
        if (r < 1 || r > g.ny - 1) continue;
        for (int f = 0; f < 2; f++) {
          double w = d[5 * f + j];
          if (iy == 1) w -= d[5 * f] * d4[j] / d4[0];
          if (iy == g.ny - 1) w -= d[5 * f + 4] * d4[j] / d4[4];
          tf[(size_t)(r + 1) * 10 + 2 * m + f] = w;
        }
      }
    tb.want(&c->derT, tb.add(t));
    tb.want(&c->derF, tb.add(tf));
    if (solve_in_lds(g)) {
      solve_table(h, g.ny, t);
      tb.want(&c->tab, tb.add(t));
    }
  }
  ScalarBlock s0;
  std::memset(&s0, 0, sizeof s0);
  s0.sc.meanpx = p->meanpx;
  s0.sc.meanpz = p->meanpz;
  const size_t scalars = tb.add(&s0, 1);
  tb.want(&c->sc, scalars);
  tb.want(&c->cfl_max, scalars + offsetof(ScalarBlock, cfl));
  tb.want(&c->stat, tb.add(std::vector<double>((size_t)10 * (g.ny + 1))));
  if ((rc = dalloc_bytes((void **)&c->tables, tb.image.size()))) return bail(rc);
  if (hipMemcpy(c->tables, tb.image.data(), tb.image.size(), hipMemcpyHostToDevice) != hipSuccess)
    return bail(fail(CHAN_E_STATE, "upload of the set-up failed"));
  tb.place(c->tables);
  // stored explicit terms start at zero (ODE3 = 0 in the first substep)
  if (hipMemset(c->old, 0, esz * 2 * (g.ny - 1) * plane) != hipSuccess ||
      hipMemset(c->V, 0, sizeof(cx<double>) * 3 * NyP) != hipSuccess)
    return bail(fail(CHAN_E_STATE, "hipMemset failed"));
  *out = c;
  return 0;
}

int chan_destroy(chan_ctx *c) {
  if (!c) return 0;
  if (c->st) hipStreamSynchronize(c->st);
  if (c->les) les_free(c->les);
  c->stage.free();
  if (c->step_row) hipHostFree(c->step_row);
  for (auto &r : c->pend) {
    hipEventDestroy(r.a);
    hipEventDestroy(r.b);
  }
  for (auto e : c->pool) hipEventDestroy(e);
  void *bufs[] = {c->V, c->old, c->rhs, c->L, c->A, c->B, c->P, c->tables, c->F0, c->gain, c->Fkeep};
  for (void *b : bufs)
    if (b) hipFree(b);
  if (c->st) hipStreamDestroy(c->st);
  setup_free(c->hs);
  delete c;
  return 0;
}

int chan_sizes(const chan_ctx *c, int32_t s[5]) {
  if (!c || !s) return fail(CHAN_E_ARG, "null argument");
  s[0] = c->g.nx;
  s[1] = c->g.ny;
  s[2] = c->g.nz;
  s[3] = c->g.nxd;
  s[4] = c->g.nzd;
  return 0;
}

int chan_get_setup(const chan_ctx *c, double *y, double *der, double *bnd) {
  if (!c) return fail(CHAN_E_ARG, "null argument");
  if (y) std::memcpy(y, c->hs.y, sizeof(double) * c->g.Ny);
  if (der) std::memcpy(der, c->hs.der, sizeof(double) * 20 * (c->g.ny - 1));
  if (bnd) std::memcpy(bnd, c->hs.bnd, sizeof(double) * 50);
  return 0;
}

int chan_setup_host(const chan_params *p, int32_t sizes[5], double *y, double *der, double *bnd, double *bc,
                    double *d0fac) {
  if (!p) return fail(CHAN_E_ARG, "null argument");
  if (p->nx < 1 || p->nz < 1 || p->ny < 8) return fail(CHAN_E_ARG, "need nx >= 1, nz >= 1, ny >= 8");
  HostSetup h;
  setup_build(h, p->nx, p->ny, p->nz, p->alfa0, p->beta0, p->a, p->ymin, p->ymax);
  if (sizes) {
    sizes[0] = p->nx;
    sizes[1] = p->ny;
    sizes[2] = p->nz;
    sizes[3] = h.nxd;
    sizes[4] = h.nzd;
  }
  if (y) std::memcpy(y, h.y, sizeof(double) * (p->ny + 3));
  if (der) std::memcpy(der, h.der, sizeof(double) * 20 * (p->ny - 1));
  if (bnd) std::memcpy(bnd, h.bnd, sizeof(double) * 50);
  if (bc) std::memcpy(bc, h.bc, sizeof(double) * 40);
  if (d0fac) std::memcpy(d0fac, h.d0fac, sizeof(double) * 5 * (p->ny + 1));
  setup_free(h);
  return 0;
}

// A host field to its device layout in V, by way of B.  Waits whatever fails: until
// then the transfer may still read the caller's buffer.
static hipError_t field_to_device(chan_ctx *c, const double *host, cx<double> *V) {
  const size_t n = (size_t)3 * c->g.npair * c->g.Ny;
  cx<double> *stage = static_cast<cx<double> *>(c->B);
  hipError_t e = copy_to_device(c->stage, stage, host, n * sizeof(cx<double>), c->st);
  if (e == hipSuccess) e = launch_to_device_layout(c->st, stage, V, c->g);
  const hipError_t end = hipStreamSynchronize(c->st);
  return e != hipSuccess ? e : end;
}

int chan_set_field(chan_ctx *c, const double *V) {
  if (!c || !V) return fail(CHAN_E_ARG, "null argument");
  HIPCHK(field_to_device(c, V, c->V));
  c->field_set = true;
  return 0;
}

int chan_get_field(chan_ctx *c, double *V) {
  if (!c || !V) return fail(CHAN_E_ARG, "null argument");
  const size_t n = (size_t)3 * c->g.npair * c->g.Ny;
  cx<double> *stage = static_cast<cx<double> *>(c->B);
  HIPCHK(launch_to_host_layout(c->st, c->V, stage, c->g));
  HIPCHK(copy_to_host(c->stage, V, stage, n * sizeof(cx<double>), c->st));
  return 0;
}

int chan_set_body_force(chan_ctx *c, const double *F) {
  if (!c) return fail(CHAN_E_ARG, "null argument");
  HIPCHK(hipStreamSynchronize(c->st));
  if (!F) {
    if (c->F0) HIPCHK(hipFree(c->F0));
    c->F0 = nullptr;
    return 0;
  }
  int rc;
  if (!c->F0 && (rc = dalloc(&c->F0, 3 * (size_t)c->g.Ny * c->g.ps))) return rc;
  HIPCHK(field_to_device(c, F, c->F0));
  return 0;
}

int chan_set_body_force_feedback(chan_ctx *c, const int32_t src[3], const double *gain) {
  if (!c) return fail(CHAN_E_ARG, "null argument");
  bool on = src && gain;
  if (on) {
    on = false;
    for (int k = 0; k < 3; k++) {
      if (src[k] < -1 || src[k] > 2) return fail(CHAN_E_ARG, "feedback source component %d of force component %d is not -1, 0, 1 or 2", src[k], k);
      on = on || src[k] >= 0;
    }
  }
  HIPCHK(hipStreamSynchronize(c->st));
  if (!on) {
    if (c->gain) HIPCHK(hipFree(c->gain));
    c->gain = nullptr;
    return 0;
  }
  const size_t n = (size_t)3 * c->g.Ny * (c->g.Nz + 1);
  int rc;
  if (!c->gain && (rc = dalloc(&c->gain, n))) return rc;
  HIPCHK(hipMemcpy(c->gain, gain, n * sizeof(double), hipMemcpyHostToDevice));
  for (int k = 0; k < 3; k++) c->src[k] = src[k];
  return 0;
}

int chan_get_body_force(chan_ctx *c, double *F) {
  if (!c || !F) return fail(CHAN_E_ARG, "null argument");
  const size_t n = (size_t)3 * c->g.npair * c->g.Ny;
  cx<double> *stage = static_cast<cx<double> *>(c->B);
  if (!c->F0 && !c->gain) {
    std::memset(F, 0, n * sizeof(cx<double>));
    return 0;
  }
  // the products buffer (dead between calls; chan_create gives it at least 48
  // bytes per point) holds the force in the device layout, 3*Ny*ps complex FP64
  cx<double> *dev = static_cast<cx<double> *>(c->P);
  ForceArgs a = force_args(c);
  a.out = dev;
  HIPCHK(launch_force(c->st, a));
  HIPCHK(launch_to_host_layout(c->st, dev, stage, c->g));
  HIPCHK(copy_to_host(c->stage, F, stage, n * sizeof(cx<double>), c->st));
  return 0;
}

int chan_keep_body_force(chan_ctx *c, int32_t on) {
  if (!c) return fail(CHAN_E_ARG, "null argument");
  HIPCHK(hipStreamSynchronize(c->st));
  c->kept_state = 0;
  if (!on) {
    if (c->Fkeep) HIPCHK(hipFree(c->Fkeep));
    c->Fkeep = nullptr;
    return 0;
  }
  int rc;
  if (!c->Fkeep && (rc = dalloc(&c->Fkeep, 3 * (size_t)c->g.Ny * c->g.ps))) return rc;
  return 0;
}

int chan_get_applied_body_force(chan_ctx *c, double *F) {
  if (!c || !F) return fail(CHAN_E_ARG, "null argument");
  if (!c->Fkeep) return fail(CHAN_E_STATE, "get_applied_body_force without keep_body_force");
  if (!c->kept_state) return fail(CHAN_E_STATE, "get_applied_body_force before a buildrhs");
  const size_t n = (size_t)3 * c->g.npair * c->g.Ny;
  if (c->kept_state == 2) {
    std::memset(F, 0, n * sizeof(cx<double>));
    return 0;
  }
  cx<double> *stage = static_cast<cx<double> *>(c->B);
  HIPCHK(launch_to_host_layout(c->st, c->Fkeep, stage, c->g));
  HIPCHK(copy_to_host(c->stage, F, stage, n * sizeof(cx<double>), c->st));
  return 0;
}

int chan_get_rhs(chan_ctx *c, double *R) {
  if (!c || !R) return fail(CHAN_E_ARG, "null argument");
  // rhs is [2][ny-1][ps]: the same transpose as the field with ny-1 rows
  Geom g = c->g;
  g.Ny = g.ny - 1;
  cx<double> *stage = static_cast<cx<double> *>(c->B);
  for (int k = 0; k < 2; k++) {
    Geom g1 = g;
    // one component at a time: the transpose kernel runs over 3 components,
    // so reuse it with a single-component view
    dim3 grid((unsigned)((g1.npair + 31) / 32), (unsigned)((g1.Ny + 31) / 32), 1);
    hipLaunchKernelGGL(k_to_host, grid, dim3(32, 8), 0, c->st, c->rhs + (size_t)k * g1.Ny * g1.ps,
                       stage + (size_t)k * g1.npair * g1.Ny, g1);
    HIPCHK(hipGetLastError());
  }
  HIPCHK(copy_to_host(c->stage, R, stage, sizeof(cx<double>) * 2 * (size_t)g.npair * g.Ny, c->st));
  return 0;
}

int chan_get_scalars(chan_ctx *c, chan_scalars *s) {
  if (!c || !s) return fail(CHAN_E_ARG, "null argument");
  ScalarBlock b;
  HIPCHK(hipMemcpyAsync(&b, c->sc, sizeof b, hipMemcpyDeviceToHost, c->st));
  HIPCHK(hipStreamSynchronize(c->st));
  DevScalars &d = b.sc;
  for (int k = 0; k < CFL_SLOTS; k++) d.cfl_bits = std::max(d.cfl_bits, b.cfl[k * CFL_STRIDE]);
  s->time = c->time;
  s->deltat = c->deltat;
  s->meanpx = d.meanpx;
  s->meanpz = d.meanpz;
  s->corrpx = d.corrpx;
  s->corrpz = d.corrpz;
  s->fr[0] = d.fr[0];
  s->fr[1] = d.fr[1];
  s->fr[2] = d.fr[2];
  s->cfl = cfl_value(d);
  return 0;
}

int chan_set_scalars(chan_ctx *c, const chan_scalars *s) {
  if (!c || !s) return fail(CHAN_E_ARG, "null argument");
  ScalarBlock b;
  std::memset(&b, 0, sizeof b);
  DevScalars &d = b.sc;
  d.meanpx = s->meanpx;
  d.meanpz = s->meanpz;
  d.corrpx = s->corrpx;
  d.corrpz = s->corrpz;
  d.fr[0] = s->fr[0];
  d.fr[1] = s->fr[1];
  d.fr[2] = s->fr[2];
  const double cf = s->cfl < 0 ? 0.0 : s->cfl;
  std::memcpy(&d.cfl_bits, &cf, sizeof cf);
  c->time = s->time;
  c->deltat = s->deltat;
  HIPCHK(hipMemcpyAsync(c->sc, &b, sizeof b, hipMemcpyHostToDevice, c->st));
  HIPCHK(hipStreamSynchronize(c->st));
  return 0;
}

extern "C++" {
// K1-K3 with transform arithmetic and intermediates in R (double, or float
// in the split mode)
template <typename R>
static int products_t(chan_ctx *c, int plane0, int nplanes, bool prods, int cfl) {
  // the physical grid where a CFL maximum is taken over it, else the alias-free one
  const bool small = prods && !cfl;
  Geom g = c->g;
  const HostSetup &h = c->hs;
  const int M = small ? c->mxs : 2 * g.nxd;
  if (small) g.nzd = c->nzs;
  // the transform kernels index A and B from the launch's first plane: the
  // base pointers are offset so that every plane keeps its own slices
  const size_t slab = (size_t)g.nzd * g.Nx;
  cx<R> *A = static_cast<cx<R> *>(c->A) + (size_t)plane0 * 3 * slab;
  cx<R> *B = static_cast<cx<R> *>(c->B) + (size_t)plane0 * NPROD * slab;
  cx<R> *P = static_cast<cx<R> *>(c->P);
  const cx<R> *twz = static_cast<const cx<R> *>(small ? c->twzs : c->twz);
  const cx<R> *twx = static_cast<const cx<R> *>(small ? c->twxs : c->twx);
  const R factor = small ? (R)(1.0 / ((double)M * g.nzd)) : (R)h.factor;
  int rc;
  if ((rc = timed(c, small ? "zinv" : "zinv_cfl", [&] { return launch_zinv<R>(g.nzd, c->st, c->V, A, twz, g, plane0, nplanes); }))) return rc;
  if ((rc = timed(c, small ? "xpass" : (prods ? "xpass_cfl" : "cfl"), [&] {
         return launch_xpass<R>(M, c->st, A, B, twx, g, plane0, nplanes, prods, cfl, c->dy, h.dx, h.dz, factor,
                                c->cfl_max);
       })))
    return rc;
  if (prods)
    if ((rc = timed(c, small ? "zfwd" : "zfwd_cfl", [&] { return launch_zfwd<R>(g.nzd, c->st, B, P, twz, g, plane0, nplanes); }))) return rc;
  return 0;
}

static int products(chan_ctx *c, int plane0, int nplanes, bool prods, int cfl) {
  return c->split ? products_t<float>(c, plane0, nplanes, prods, cfl) : products_t<double>(c, plane0, nplanes, prods, cfl);
}

template <typename R>
static int rhs_t(chan_ctx *c, const double ode[3], bool keep, bool store_old) {
  RhsArgs<R> a;
  a.P = static_cast<const cx<R> *>(c->P);
  a.V = c->V;
  a.old = static_cast<cx<R> *>(c->old);
  a.rhs = c->rhs;
  a.derT = c->derT;
  a.sc = c->sc;
  a.store_old = store_old;
  a.g = c->g;
  a.ode0 = ode[0];
  a.ode1 = ode[1];
  a.ode2 = ode[2];
  a.dt = c->deltat;
  a.ni = c->prm.ni;
  a.chunk = 0;
  const bool force = c->F0 || c->gain;
  if (keep) c->kept_state = force ? 1 : 2;
  ForceArgs f = force_args(c);
  if (force && keep) {
    f.out = c->Fkeep;
    int rc;
    if ((rc = timed(c, "force_keep", [&] { return launch_force(c->st, f); }))) return rc;
  }
  return timed(c, "rhs", [&] { return launch_rhs<R>(c->st, a, force ? &f : nullptr); });
}

// keep: store the applied force when keeping is on (chan_step asks only in
// its last substep, whose force is the one that stays).  store_old: leave the
// explicit terms behind for a following substep with ode[2] != 0.
static int buildrhs(chan_ctx *c, const double ode[3], bool compute_cfl, bool keep, bool store_old) {
  const Geom &g = c->g;
  int rc;
  if ((rc = products(c, 0, g.Ny, true, compute_cfl ? 1 : 0))) return rc;
  keep = keep && c->Fkeep;
  return c->split ? rhs_t<float>(c, ode, keep, store_old) : rhs_t<double>(c, ode, keep, store_old);
}
}  // extern "C++"

int chan_buildrhs(chan_ctx *c, const double ode[3], int32_t compute_cfl) {
  if (!c || !ode) return fail(CHAN_E_ARG, "null argument");
  if (!c->field_set) return fail(CHAN_E_STATE, "buildrhs before set_field");
  return buildrhs(c, ode, compute_cfl != 0, true, true);
}

int chan_linsolve(chan_ctx *c, double lambda) {
  if (!c) return fail(CHAN_E_ARG, "null argument");
  if (!c->field_set) return fail(CHAN_E_STATE, "linsolve before set_field");
  const Geom &g = c->g;
  int rc;
  SolveArgs s;
  s.V = c->V;
  s.rhs = c->rhs;
  s.L = c->L;
  s.der = c->der;
  std::memcpy(s.bc, c->hs.bc, sizeof s.bc);
  for (int k = 0; k < 2; k++) {
    const double *lw = c->hs.bc[k ? BC_V0 : BC_ETA0], *lg = c->hs.bc[k ? BC_V0M1 : BC_ETA0M1];
    const double *hw = c->hs.bc[k ? BC_VN : BC_ETAN], *hg = c->hs.bc[k ? BC_VNP1 : BC_ETANP1];
    for (int j = 0; j < 5; j++) {
      s.wall[k].lo_ghost[j] = lg[j] / lg[0];
      s.wall[k].lo_wall[j] = lw[j] / lw[1];
      s.wall[k].hi_ghost[j] = hg[j] / hg[4];
      s.wall[k].hi_wall[j] = hw[j] / hw[3];
    }
  }
  s.g = g;
  s.lambda = lambda;
  s.ni = c->prm.ni;
  s.u0 = c->prm.u0;
  s.uN = c->prm.uN;
  UwArgs u;
  u.V = c->V;
  u.tab = c->tab;
  u.der = c->der;
  u.d0fac = c->d0fac;
  std::memcpy(u.bnd, c->hs.bnd, sizeof u.bnd);
  u.g = g;
  const bool lds = solve_in_lds(g);
  if ((rc = lds ? timed(c, "solve_lds", [&] { return launch_solve_lds(c->st, s, u); })
                : timed(c, "solve_ve", [&] { return launch_solve(c->st, s); })))
    return rc;
  MeanArgs m;
  m.V = c->V;
  m.y = c->y;
  m.sc = c->sc;
  std::memcpy(m.bc, c->hs.bc, sizeof m.bc);
  m.g = g;
  m.meanflowx = c->prm.meanflowx;
  m.meanflowz = c->prm.meanflowz;
  m.gamma = c->prm.gamma;
  m.ni = c->prm.ni;
  m.cpi = c->prm.cpi;
  m.cpi_type = c->prm.cpi_type;
  if ((rc = timed(c, "mean", [&] { return launch_mean(c->st, m); }))) return rc;
  return lds ? 0 : timed(c, "uw", [&] { return launch_uw(c->st, u); });
}

int chan_initial(chan_ctx *c) {
  if (!c) return fail(CHAN_E_ARG, "null argument");
  if (!c->field_set) return fail(CHAN_E_STATE, "initial before set_field");
  if (c->deltat == 0) c->deltat = 1.0;
  const Geom &g = c->g;
  int rc;
  // interior planes iy = 1..ny-1 are plane indices 2..ny
  if ((rc = products(c, 2, g.ny - 1, false, 1))) return rc;
  MeanArgs m;
  std::memset(&m, 0, sizeof m);
  m.V = c->V;
  m.y = c->y;
  m.sc = c->sc;
  m.g = g;
  m.gamma = c->prm.gamma;
  m.ni = c->prm.ni;
  m.cpi = c->prm.cpi;
  m.cpi_type = c->prm.cpi_type;
  return timed(c, "flowrate", [&] { return launch_flowrate(c->st, m); });
}

int chan_stats(chan_ctx *c, const double *avg, double *out) {
  if (!c || !out) return fail(CHAN_E_ARG, "null argument");
  if (!c->field_set) return fail(CHAN_E_STATE, "stats before set_field");
  const Geom &g = c->g;
  const size_t n1 = (size_t)g.ny + 1;
  double *dav = nullptr;
  if (avg) {
    dav = c->stat;
    HIPCHK(hipMemcpyAsync(dav, avg, sizeof(double) * 3 * n1, hipMemcpyHostToDevice, c->st));
  }
  int rc;
  if ((rc = timed(c, "stats", [&] { return launch_stats(c->st, c->V, dav, c->stat + 3 * n1, g); }))) return rc;
  HIPCHK(hipMemcpyAsync(out, c->stat + 3 * n1, sizeof(double) * 7 * n1, hipMemcpyDeviceToHost, c->st));
  HIPCHK(hipStreamSynchronize(c->st));
  return 0;
}

int chan_outstats(chan_ctx *c, double row[11]) {
  if (!c || !row) return fail(CHAN_E_ARG, "null argument");
  const Geom &g = c->g;
  // one kernel writes the rows and scalars and resets the running CFL maximum
  // (cfl=0 in outstats)
  StepRow *const row0 = static_cast<StepRow *>(c->step_row);
  hipLaunchKernelGGL(k_step_row, dim3(1), dim3(64), 0, c->st, c->V, row0, c->sc, c->cfl_max, g);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(c->st));
  const StepRow s = *row0;
  const DevScalars &d = s.sc;
  const double rg = cfl_value(d);
  if (!std::isfinite(rg)) return fail(CHAN_E_NOTFINITE, "CFL maximum is not finite (%g): the field holds NaN or Inf", rg);
  if (c->prm.cflmax > 0) c->deltat = c->prm.cflmax / rg;
  const double *b140 = c->hs.bnd[B_D140], *b14n = c->hs.bnd[B_D14N];
  double d11 = 0, d21 = 0, d12 = 0, d22 = 0;
  for (int j = 0; j < 5; j++) {
    d12 += b14n[j] * s.hi[0][j];
    d22 += b14n[j] * s.hi[1][j];
  }
  d12 = -d12;
  d22 = -d22;
  for (int j = 0; j < 5; j++) {
    d11 += b140[j] * s.lo[0][j];
    d21 += b140[j] * s.lo[1][j];
  }
  row[0] = c->time;
  row[1] = d11;
  row[2] = d12;
  row[3] = d21;
  row[4] = d22;
  row[5] = d.fr[0] + d.corrpx * d.fr[2];
  row[6] = d.meanpx + d.corrpx;
  row[7] = d.fr[1] + d.corrpz * d.fr[2];
  row[8] = d.meanpz + d.corrpz;
  row[9] = rg * c->deltat;
  row[10] = c->deltat;
  return 0;
}

// One time step.  store_old: also leave the third substep's explicit terms
// behind; a following step's first substep (ode[2] = 0) does not read them.
static int time_step(chan_ctx *c, double row[11], bool store_old) {
  int rc;
  const double *ode[3] = {RK1, RK2, RK3};
  for (int k = 0; k < 3; k++) {
    c->time = c->time + 2.0 / ode[k][0] * c->deltat;
    if (!c->field_set) return fail(CHAN_E_STATE, "step before set_field");
    if ((rc = buildrhs(c, ode[k], k == 2, k == 2, k < 2 || store_old))) return rc;
    if ((rc = chan_linsolve(c, ode[k][0] / c->deltat))) return rc;
  }
  return chan_outstats(c, row);
}

int chan_step(chan_ctx *c, double row[11]) {
  if (!c || !row) return fail(CHAN_E_ARG, "null argument");
  return time_step(c, row, true);
}

int chan_steps(chan_ctx *c, int32_t n, double *rows) {
  if (!c || (n > 0 && !rows)) return fail(CHAN_E_ARG, "null argument");
  for (int32_t i = 0; i < n; i++) {
    int rc = time_step(c, rows + 11 * (size_t)i, i + 1 == n);
    if (rc) return rc;
  }
  return 0;
}

int chan_timing(chan_ctx *c, int32_t enable) {
  if (!c) return fail(CHAN_E_ARG, "null argument");
  if (!enable) {
    int rc = harvest(c);
    if (rc) return rc;
  }
  c->timing = enable != 0;
  if (enable) {
    int rc = harvest(c);
    if (rc) return rc;
    for (size_t i = 0; i < c->names.size(); i++) {
      c->counts[i] = 0;
      c->ms[i] = 0;
    }
  }
  return 0;
}

int chan_kernel_times(chan_ctx *c, int32_t cap, char *names, int64_t *counts, double *total_ms, int32_t *n) {
  if (!c || !n) return fail(CHAN_E_ARG, "null argument");
  int rc = harvest(c);
  if (rc) return rc;
  *n = (int32_t)c->names.size();
  for (int32_t i = 0; i < *n && i < cap; i++) {
    if (names) {
      std::strncpy(names + 32 * i, c->names[i].c_str(), 31);
      names[32 * i + 31] = 0;
    }
    if (counts) counts[i] = c->counts[i];
    if (total_ms) total_ms[i] = c->ms[i];
  }
  return 0;
}

int chan_sync(chan_ctx *c) {
  if (!c) return fail(CHAN_E_ARG, "null argument");
  HIPCHK(hipStreamSynchronize(c->st));
  return 0;
}

int chan_fft_selftest(int32_t n, int32_t sign, int32_t batch, double *inout) {
  if (!inout || batch < 1 || (sign != 1 && sign != -1)) return fail(CHAN_E_ARG, "bad argument");
  if (!fft_size_supported(n)) return fail(CHAN_E_SIZE, "size %d not supported", n);
  std::vector<cx<double>> tw;
  twiddles(tw, n);
  cx<double> *d = nullptr, *t = nullptr;
  const size_t bytes = sizeof(cx<double>) * (size_t)n * batch;
  HIPCHK(hipMalloc(&d, bytes));
  hipError_t e = hipMalloc(&t, sizeof(cx<double>) * tw.size());
  if (e == hipSuccess) e = hipMemcpy(d, inout, bytes, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(t, tw.data(), sizeof(cx<double>) * tw.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = launch_fft_test(n, sign, 0, d, t, batch);
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemcpy(inout, d, bytes, hipMemcpyDeviceToHost);
  hipFree(d);
  if (t) hipFree(t);
  if (e != hipSuccess) return fail((int)e, "fft selftest: %s", hipGetErrorString(e));
  return 0;
}

int chan_fft768_fs_test(int32_t sign, int32_t batch, int32_t inner, int32_t reps, double *inout, double *ms) {
  if (!inout || !ms || batch < 1 || reps < 1 || inner < 1 || inner > 8 || (sign != 1 && sign != -1))
    return fail(CHAN_E_ARG, "bad argument");
  cx<double> tw[fft::FS_TW];
  fft::build_fs768_twiddles(tw);
  const size_t bytes = sizeof(cx<double>) * 768 * (size_t)batch;
  cx<double> *a = nullptr, *b = nullptr, *t = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  HIPCHK(hipMalloc(&a, bytes));
  hipError_t e = hipMalloc(&b, bytes);
  if (e == hipSuccess) e = hipMalloc(&t, sizeof tw);
  if (e == hipSuccess) e = hipMemcpy(a, inout, bytes, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(t, tw, sizeof tw, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipEventCreate(&e0);
  if (e == hipSuccess) e = hipEventCreate(&e1);
  if (e == hipSuccess) e = launch_fs768_test(a, b, t, batch, sign, 1);
  if (e == hipSuccess) e = hipMemcpy(inout, b, bytes, hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipEventRecord(e0, 0);
  for (int r = 0; r < reps && e == hipSuccess; r++) e = launch_fs768_test(a, b, t, batch, sign, inner);
  if (e == hipSuccess) e = hipEventRecord(e1, 0);
  if (e == hipSuccess) e = hipEventSynchronize(e1);
  float ft = 0;
  if (e == hipSuccess) e = hipEventElapsedTime(&ft, e0, e1);
  *ms = ft / reps;
  if (e0) hipEventDestroy(e0);
  if (e1) hipEventDestroy(e1);
  hipFree(a);
  if (b) hipFree(b);
  if (t) hipFree(t);
  if (e != hipSuccess) return fail((int)e, "chan_fft768_fs_test: %s", hipGetErrorString(e));
  return 0;
}

int chan_fft_bench(int32_t n, int32_t sign, int32_t batch, int32_t variant, int32_t reps, double *inout, double *ms) {
  const int inner = 1 + (variant >> 4);  // transforms per load/store pair
  if (!inout || !ms || batch < 1 || reps < 1 || variant < 0 || inner > 64 || (sign != 1 && sign != -1))
    return fail(CHAN_E_ARG, "bad argument");
  if (n != 384 && n != 768 && n != 1536) return fail(CHAN_E_SIZE, "size %d not benchmarked", n);
  std::vector<cx<double>> tw;
  twiddles(tw, n);
  const size_t bytes = sizeof(cx<double>) * (size_t)n * batch;
  cx<double> *a = nullptr, *b = nullptr, *t = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  HIPCHK(hipMalloc(&a, bytes));
  hipError_t e = hipMalloc(&b, bytes);
  if (e == hipSuccess) e = hipMalloc(&t, sizeof(cx<double>) * tw.size());
  if (e == hipSuccess) e = hipMemcpy(a, inout, bytes, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(t, tw.data(), sizeof(cx<double>) * tw.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipEventCreate(&e0);
  if (e == hipSuccess) e = hipEventCreate(&e1);
  if (e == hipSuccess) e = launch_fft_bench(n, sign, variant & 15, a, b, t, batch, 1);
  if (e == hipSuccess) e = hipEventRecord(e0, 0);
  for (int r = 0; r < reps && e == hipSuccess; r++) e = launch_fft_bench(n, sign, variant & 15, a, b, t, batch, inner);
  if (e == hipSuccess) e = hipEventRecord(e1, 0);
  if (e == hipSuccess) e = hipEventSynchronize(e1);
  float ft = 0;
  if (e == hipSuccess) e = hipEventElapsedTime(&ft, e0, e1);
  if (e == hipSuccess) e = hipMemcpy(inout, b, bytes, hipMemcpyDeviceToHost);
  *ms = ft / reps;
  if (e0) hipEventDestroy(e0);
  if (e1) hipEventDestroy(e1);
  hipFree(a);
  if (b) hipFree(b);
  if (t) hipFree(t);
  if (e != hipSuccess) return fail((int)e, "fft bench: %s", hipGetErrorString(e));
  return 0;
}

int chan_copy_selftest(int64_t bytes, int32_t reps, double *ms) {
  if (bytes <= 0 || bytes % 32 != 0 || reps < 1 || !ms) return fail(CHAN_E_ARG, "bad argument");
  double4 *a = nullptr, *b = nullptr;
  const size_t n = (size_t)bytes / sizeof(double4);
  HIPCHK(hipMalloc(&a, n * sizeof(double4)));
  hipError_t e = hipMalloc(&b, n * sizeof(double4));
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (e == hipSuccess) e = hipMemset(a, 0, n * sizeof(double4));
  if (e == hipSuccess) e = hipEventCreate(&e0);
  if (e == hipSuccess) e = hipEventCreate(&e1);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_copy, dim3(2048), dim3(256), 0, 0, a, b, n);  // warm-up
    e = hipEventRecord(e0, 0);
  }
  for (int r = 0; r < reps && e == hipSuccess; r++) {
    hipLaunchKernelGGL(k_copy, dim3(2048), dim3(256), 0, 0, a, b, n);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipEventRecord(e1, 0);
  if (e == hipSuccess) e = hipEventSynchronize(e1);
  float t = 0;
  if (e == hipSuccess) e = hipEventElapsedTime(&t, e0, e1);
  *ms = t / reps;
  if (e0) hipEventDestroy(e0);
  if (e1) hipEventDestroy(e1);
  hipFree(a);
  if (b) hipFree(b);
  if (e != hipSuccess) return fail((int)e, "copy selftest: %s", hipGetErrorString(e));
  return 0;
}

}  // extern "C"
