// k_mlp.hip -- the learned subgrid-stress closure: an MLP 46 -> 64 -> 64 ->
// 64 -> 6 (ReLU) with BF16 weights and activations and FP32 accumulation on
// the CDNA4 matrix cores (v_mfma_f32_16x16x32_bf16).  The reference has no
// counterpart; the network maps box-filtered velocity gradients to the six
// subgrid stresses.
//
// Matrix-core fragments (16x16x32, one wavefront, lane l, q = l / 16):
//   A (16 x 32): A[l % 16][8 q + j], j = 0..7
//   B (32 x 16): B[8 q + j][l % 16]
//   D (16 x 16): D[4 q + i][l % 16], i = 0..3
// Samples sit in the columns (B and D), units in the rows: a layer is D =
// W^T B with the weights as A fragments, which a wave keeps in registers for
// all its samples, and four swaps of register pairs with lane rows turn the D
// layout of one layer into the B layout of the next (next_operand), so that
// activations never leave the registers between layers.  Layers are padded to
// 64 inputs (46 features + zeros) and 16 outputs (6 + zeros).  Weights are kept
// twice in BF16: Woi[l][out][in] feeds the forward pass (8 consecutive inputs
// per lane), Wio[l][in][out] the backward data pass; biases stay FP32.
//
// Kernels: k_mlp_fwd, k_mlp_fwd_les (inference from BF16 or FP32 rows, from the
// closure's gradients), k_mlp_grad (forward, backward and weight gradients of a minibatch
// in one pass, per-block partial sums) and k_mlp_update (sums the partials in a
// fixed order, then Adam on the FP32 master weights, refreshing the BF16 copies).
#include "chan_internal.hpp"
#include "mlp_internal.hpp"

namespace chan {
namespace mlp {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

__device__ __forceinline__ f32x4 mma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x8 load8(const __bf16 *p) { return *reinterpret_cast<const bf16x8 *>(p); }
__device__ __forceinline__ bf16x8 zero8() {
  bf16x8 z;
#pragma unroll
  for (int j = 0; j < 8; j++) z[j] = (__bf16)0.0f;
  return z;
}

// The next layer's B fragments from this layer's outputs: P[mt][h] packs the
// outputs mt*16 + 4q + 2h, + 1 of the lane's sample.  Lane row q needs the units
// ks*32 + 8q + j, which lane rows 2 (q & 1) + (j >> 2) hold for mt = 2 ks + (q >> 1):
// exchanging the register pair with the upper half of the wave and then with the
// odd rows puts them there.
__device__ __forceinline__ void next_operand(const unsigned (&P)[4][2], bf16x8 (&b)[2]) {
#pragma unroll
  for (int ks = 0; ks < 2; ks++) {
    unsigned r[4];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const auto u = __builtin_amdgcn_permlane32_swap(P[2 * ks][h], P[2 * ks + 1][h], false, false);
      const auto v = __builtin_amdgcn_permlane16_swap(u[0], u[1], false, false);
      r[h] = v[0];
      r[2 + h] = v[1];
    }
    __builtin_memcpy(&b[ks], r, sizeof r);
  }
}

__device__ __forceinline__ unsigned pack2(__bf16 x, __bf16 y) {
  unsigned short u, v;
  __builtin_memcpy(&u, &x, 2);
  __builtin_memcpy(&v, &y, 2);
  return (unsigned)u | (unsigned)v << 16;
}

// The weights of the forward pass as A fragments, 104 registers, and the biases
// in LDS.
constexpr int WROW = 72;  // BF16 values per unit's row of weights in LDS, padded
struct Layers {
  bf16x8 h[3][4][2], o[2];
  __device__ __forceinline__ void load(const Weights &w, int c16, int q) {
#pragma unroll
    for (int L = 0; L < 3; L++)
#pragma unroll
      for (int mt = 0; mt < 4; mt++)
#pragma unroll
        for (int ks = 0; ks < 2; ks++) h[L][mt][ks] = load8(w.woi + WOFF[L] + (mt * 16 + c16) * KP + ks * 32 + 8 * q);
#pragma unroll
    for (int ks = 0; ks < 2; ks++) o[ks] = load8(w.woi + WOFF[3] + c16 * KP + ks * 32 + 8 * q);
  }
  // the same from rows of WROW values
  __device__ __forceinline__ void load_rows(const __bf16 *r, int c16, int q) {
#pragma unroll
    for (int L = 0; L < 3; L++)
#pragma unroll
      for (int mt = 0; mt < 4; mt++)
#pragma unroll
        for (int ks = 0; ks < 2; ks++) h[L][mt][ks] = load8(r + (L * H + mt * 16 + c16) * WROW + ks * 32 + 8 * q);
#pragma unroll
    for (int ks = 0; ks < 2; ks++) o[ks] = load8(r + (3 * H + c16) * WROW + ks * 32 + 8 * q);
  }
};

// z of one hidden layer: D tile mt of W^T b, plus bias
__device__ __forceinline__ f32x4 dense(const bf16x8 (&A)[2], const bf16x8 (&b)[2]) {
  f32x4 acc = {0, 0, 0, 0};
  acc = mma(A[0], b[0], acc);
  return mma(A[1], b[1], acc);
}
__device__ __forceinline__ f32x4 bias4(const float *b) { return *reinterpret_cast<const f32x4 *>(b); }

// Output of one 16-sample tile from its B fragments: lane (q, c16) returns
// y[4q + i] of sample c16.
__device__ __forceinline__ f32x4 forward_tile(const Layers &W, const float *bias, bf16x8 (&b)[2], int q) {
#pragma unroll
  for (int L = 0; L < 3; L++) {
    unsigned P[4][2];
#pragma unroll
    for (int mt = 0; mt < 4; mt++) {
      const f32x4 acc = dense(W.h[L][mt], b), bb = bias4(bias + BOFF[L] + mt * 16 + 4 * q);
      __bf16 v[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float z = acc[i] + bb[i];
        v[i] = (__bf16)(z > 0.0f ? z : 0.0f);
      }
      P[mt][0] = pack2(v[0], v[1]);
      P[mt][1] = pack2(v[2], v[3]);
    }
    next_operand(P, b);
  }
  return dense(W.o, b) + bias4(bias + BOFF[3] + 4 * q);
}
__device__ __forceinline__ void store_tile(float *__restrict__ Y, const f32x4 &y, int row, int n, int q) {
  if (row >= n) return;
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (4 * q + i < OUT) Y[(size_t)row * OUT + 4 * q + i] = y[i];
}

// ------------------------------------------------------------ forward --
// Sources of input rows: raw(row) starts the loads of lane row q's features of a
// sample, operand(raw) forms its B fragments.
struct FromBf16 {  // BF16 rows [n][64]
  const __bf16 *X;
  struct Raw {
    bf16x8 v[2];
  };
  __device__ __forceinline__ Raw raw(int row, int q) const {
    return Raw{{load8(X + (size_t)row * KP + 8 * q), load8(X + (size_t)row * KP + 32 + 8 * q)}};
  }
  __device__ __forceinline__ void operand(const Raw &r, bf16x8 (&b)[2]) const {
    b[0] = r.v[0];
    b[1] = r.v[1];
  }
};
struct FromFloat {  // FP32 rows [n][46], any alignment of a float
  const float *X;
  struct Raw {
    float v[2][8];
  };
  __device__ __forceinline__ Raw raw(int row, int q) const {
    Raw r;
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int f = 32 * k + 8 * q + j;
        r.v[k][j] = f < IN ? X[(size_t)row * IN + f] : 0.0f;
      }
    return r;
  }
  __device__ __forceinline__ void operand(const Raw &r, bf16x8 (&b)[2]) const {
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int j = 0; j < 8; j++) b[k][j] = (__bf16)r.v[k][j];
  }
};

// y [N][6] of 16-sample tiles, one wave each, the weights in registers.  A block's
// waves fetch them together, by way of LDS, while the first rows are on their way: each for
// itself, the waves spend most of a short call on that (us for 1024, 32768, 65536 and 599040
// BF16 rows: 5.3, 8.7, 10.3 and 34.5; together 3.6, 4.8, 6.3 and 31.4).  With the
// weights read from LDS per tile and the activations turned through LDS
// between layers it was 4.6, 6.0, 8.8 and 54.7.
template <class Src>
__global__ __launch_bounds__(256, 2) void k_mlp_fwd(Weights w, Src src, int n, float *__restrict__ Y) {
  __shared__ __align__(16) float bias[BSIZE];
  __shared__ __align__(16) __bf16 wl[WSIZE / KP * WROW];
  const int wv = threadIdx.x / 64, l = threadIdx.x % 64, c16 = l % 16, q = l / 16;
  const int ntile = (n + 15) / 16, stride = gridDim.x * 4;
  int tt = blockIdx.x * 4 + wv;
  auto next = src.raw(min(tt * 16 + c16, n - 1), q);
#pragma unroll
  for (int k = 0; k < (WSIZE / 8 + 255) / 256; k++) {
    const int i = threadIdx.x + 256 * k;
    if (i < WSIZE / 8) *reinterpret_cast<bf16x8 *>(wl + i / (KP / 8) * WROW + i % (KP / 8) * 8) = load8(w.woi + 8 * i);
  }
  for (int i = threadIdx.x; i < BSIZE; i += 256) bias[i] = w.bias[i];
  __syncthreads();
  Layers W;
  W.load_rows(wl, c16, q);
  if (tt >= ntile) return;
  for (; tt < ntile; tt += stride) {
    const auto cur = next;
    next = src.raw(min((tt + stride) * 16 + c16, n - 1), q);  // rows past n read row n-1
    bf16x8 b[2];
    src.operand(cur, b);
    store_tile(Y, forward_tile(W, bias, b, q), tt * 16 + c16, n, q);
  }
}

// The same for the closure's normalised features, formed straight from the
// velocity gradients G[9][n] (LesSource): feature 9 k + j of a sample is gradient
// j of the row dy[k] = 0, -2, -1, 1, 2 away (clamped to 0..ny), the last one y+.
// A wave takes 64 samples, one per lane, so that every load is contiguous and
// the means and scales are wave-uniform, and turns them into fragments through
// LDS.  (x - mean) / scale is what the division gives: one product with the
// rounded reciprocal and one exact-remainder correction where nothing can overflow or
// lose bits in them (Markstein's theorem), which is where x - mean is zero or of a size in
// [SPAN_X^-1, SPAN_X] and every scale is in [SPAN_D^-1, SPAN_D] (LesSource::quick);
// a wave with a sample outside divides.  599040 samples take 42 us, 50 with divisions
// throughout.
constexpr int FROW = 72;  // BF16 values per sample in LDS, padded
constexpr float SPAN_X = 0x1p100f;
__device__ __forceinline__ unsigned bits_of(float x) { return __float_as_uint(x); }
__global__ __launch_bounds__(256, 2) void k_mlp_fwd_les(Weights w, LesSource s, const float *__restrict__ norm,
                                                        const double *__restrict__ yplus, float *__restrict__ Y) {
  __shared__ __align__(16) float bias[BSIZE];
  __shared__ __align__(16) __bf16 rows[4][64 * FROW];
  for (int i = threadIdx.x; i < BSIZE; i += 256) bias[i] = w.bias[i];
  const int wv = threadIdx.x / 64, l = threadIdx.x % 64, c16 = l % 16, q = l / 16, n = s.n;
  const int ngrp = (n + 63) / 64, stride = gridDim.x * 4;
  Layers W;
  W.load(w, c16, q);
  __syncthreads();
  int grp = blockIdx.x * 4 + wv;
  if (grp >= ngrp) return;
  __bf16 *mine = rows[wv] + l * FROW;
  float f[IN];
  auto fetch = [&](int g) {
    const int sm = min(g * 64 + l, n - 1), iy = sm / s.plane, o = sm - iy * s.plane;
    const int dy[5] = {0, -2, -1, 1, 2};
#pragma unroll
    for (int k = 0; k < 5; k++) {
      const int at = min(max(iy + dy[k], 0), s.ny) * s.plane + o;
#pragma unroll
      for (int j = 0; j < 9; j++) f[9 * k + j] = s.G[(size_t)j * n + at];
    }
    f[IN - 1] = (float)yplus[iy];
  };
  for (; grp < ngrp; grp += stride) {
    fetch(grp);
    float hi = 0.0f;          // largest |x - mean|
    unsigned lo = ~0u;        // smallest one that is not zero: its bits shifted left, less one
#pragma unroll
    for (int k = 0; k < IN; k++) {
      f[k] -= norm[k];
      hi = fmaxf(hi, fabsf(f[k]));
      lo = min(lo, (bits_of(f[k]) << 1) - 1u);
    }
    auto put = [&](auto quotient) {
#pragma unroll
      for (int c = 0; c < 8; c++) {
        bf16x8 v = zero8();
#pragma unroll
        for (int j = 0; j < 8; j++)
          if (8 * c + j < IN) v[j] = (__bf16)quotient(8 * c + j);
        *reinterpret_cast<bf16x8 *>(mine + 8 * c) = v;
      }
    };
    if (s.quick && __all(hi <= SPAN_X && lo >= (bits_of(1.0f / SPAN_X) << 1) - 1u))
      put([&](int k) {
        const float rd = norm[NORM_RECIP + k], t = f[k] * rd;
        return fmaf(fmaf(-t, norm[IN + k], f[k]), rd, t);
      });
    else
      put([&](int k) { return f[k] / norm[IN + k]; });
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll 1
    for (int t = 0; t < 4; t++) {
      const __bf16 *r = rows[wv] + (16 * t + c16) * FROW + 8 * q;
      bf16x8 b[2] = {load8(r), load8(r + 32)};
      store_tile(Y, forward_tile(W, bias, b, q), grp * 64 + 16 * t + c16, n, q);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// ------------------------------------------------------------- gradient --
// Loss and gradient of a minibatch.  The samples are cut into chunks of C * 128
// and a chunk into four slots: slot w takes the 32-sample sets at w * 32 + 128 k.
// A slot's weight gradients accumulate on the matrix cores set after set, a
// chunk's are the sum of its slots in order, the minibatch's the sum of its
// chunks in order: this fixes every rounding, so that training does not depend on
// how the work is spread.  A block takes `per` slots of one chunk and passes over
// two sets, 64 samples, at a time: each wave runs 16 samples forward and back in
// registers, leaving inputs, activations and dz of every layer in LDS as
// [unit][sample]; then wave L adds the sets' weight gradient of layer L.  With per
// = 4 the block writes its chunk's sum, with per = 2 (few chunks: twice the blocks
// at work) each slot's.  8192 samples take 19 us in this one launch (16384: 25), where
// separate forward, three backward and four weight-gradient kernels through memory took 97.
constexpr int SP = 72;  // samples per LDS row, padded: 16-byte rows, spread over the banks
struct GradLds {
  __bf16 in[4][64 * SP];   // inputs of the layers: X, act 1..3
  __bf16 dz[3][64 * SP];   // dz of the hidden layers
  __bf16 dy[OP * SP];
  float bias[BSIZE];
  double red[4];
};
__global__ __launch_bounds__(256) void k_mlp_grad(Weights w, const __bf16 *__restrict__ X, const float *__restrict__ Tg,
                                                  int n, float inv_count, int chunk, int per,
                                                  float *__restrict__ part, double *__restrict__ loss_part) {
  extern __shared__ __align__(16) char smem[];
  GradLds &S = *reinterpret_cast<GradLds *>(smem);
  for (int i = threadIdx.x; i < BSIZE; i += 256) S.bias[i] = w.bias[i];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), l = threadIdx.x % 64, c16 = l % 16, q = l / 16;
  const int sc = wv * 16 + c16;  // the lane's sample in the group
  __syncthreads();
  const int nout = wv < 3 ? H : OP, NT = nout / 16;  // of the layer whose weight gradient this wave forms
  const __bf16 *tz = wv < 3 ? S.dz[wv] : S.dy;
  const int split = 4 / per, ch = blockIdx.x / split, w0 = (blockIdx.x % split) * per, C = chunk / 128;
  const int begin = ch * chunk, end = min(n, begin + chunk);
  f32x4 acc[4][4], g[4][4];  // of the current slot; of the chunk
#pragma unroll
  for (int mt = 0; mt < 4; mt++)
#pragma unroll
    for (int nt = 0; nt < 4; nt++) acc[mt][nt] = g[mt][nt] = f32x4{0, 0, 0, 0};
  float bacc = 0.0f, bsum = 0.0f;
  double lsum = 0.0;
  auto store = [&](const f32x4(&v)[4][4], float bias, int at) {
    float *dst = part + (size_t)at * GSIZE + GOFF[wv];
#pragma unroll
    for (int nt = 0; nt < 4; nt++) {
      if (nt >= NT) break;
#pragma unroll
      for (int mt = 0; mt < 4; mt++)
#pragma unroll
        for (int i = 0; i < 4; i++) dst[(mt * 16 + 4 * q + i) * nout + nt * 16 + c16] = v[mt][nt][i];
    }
    if (l < nout) dst[64 * nout + l] = bias;
  };
  for (int t0 = w0 * C; t0 < (w0 + per) * C; t0 += 2) {
    const int ts = t0 + (wv >> 1);  // this wave's set: slot ts / C, its set ts % C
    const int row = begin + (ts / C) * 32 + (ts % C) * 128 + (wv & 1) * 16 + c16;
    const bool valid = row < end;
    const size_t rc = (size_t)min(row, n - 1);
    Layers W;
    W.load(w, c16, q);
    bf16x8 b[2];
    b[0] = load8(X + rc * KP + 8 * q);
    b[1] = load8(X + rc * KP + 32 + 8 * q);
    float tg[4];
#pragma unroll
    for (int i = 0; i < 4; i++) tg[i] = 4 * q + i < OUT ? Tg[rc * OUT + 4 * q + i] : 0.0f;
#pragma unroll
    for (int ks = 0; ks < 2; ks++)
#pragma unroll
      for (int j = 0; j < 8; j++) S.in[0][(ks * 32 + 8 * q + j) * SP + sc] = b[ks][j];
    unsigned mask[3];
#pragma unroll
    for (int L = 0; L < 3; L++) {
      unsigned P[4][2];
      mask[L] = 0;
#pragma unroll
      for (int mt = 0; mt < 4; mt++) {
        const f32x4 h = dense(W.h[L][mt], b), bb = bias4(S.bias + BOFF[L] + mt * 16 + 4 * q);
        __bf16 v[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float z = h[i] + bb[i];
          v[i] = (__bf16)(z > 0.0f ? z : 0.0f);
          mask[L] |= (float)v[i] > 0.0f ? 1u << (4 * mt + i) : 0u;
          S.in[L + 1][(mt * 16 + 4 * q + i) * SP + sc] = v[i];
        }
        P[mt][0] = pack2(v[0], v[1]);
        P[mt][1] = pack2(v[2], v[3]);
      }
      next_operand(P, b);
    }
    {
      const f32x4 o = dense(W.o, b), bb = bias4(S.bias + BOFF[3] + 4 * q);
      __bf16 dv[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        float d = o[i] + bb[i] - tg[i];
        if (!valid || 4 * q + i >= OUT) d = 0.0f;
        lsum += (double)d * d;
        dv[i] = (__bf16)(2.0f * d * inv_count);
        S.dy[(4 * q + i) * SP + sc] = dv[i];
      }
      // dy as a B fragment: only the outputs 0..7, lane row 0, are not zero
      const unsigned p0 = pack2(dv[0], dv[1]), p1 = pack2(dv[2], dv[3]);
      unsigned r[4] = {p0, p1, (unsigned)__shfl((int)p0, c16 + 16, 64), (unsigned)__shfl((int)p1, c16 + 16, 64)};
#pragma unroll
      for (int k = 0; k < 4; k++)
        if (q) r[k] = 0;
      __builtin_memcpy(&b[0], r, sizeof r);
    }
    // back: dh = W dz_next, masked by the activation
#pragma unroll
    for (int L = 2; L >= 0; L--) {
      unsigned P[4][2];
#pragma unroll
      for (int mt = 0; mt < 4; mt++) {
        f32x4 h = {0, 0, 0, 0};
        const __bf16 *A = w.wio + WOFF[L + 1] + (size_t)(mt * 16 + c16) * (L == 2 ? OP : H);
        if (L == 2) {
          h = mma(q < 2 ? load8(A + 8 * q) : zero8(), b[0], h);
        } else {
          h = mma(load8(A + 8 * q), b[0], h);
          h = mma(load8(A + 32 + 8 * q), b[1], h);
        }
        __bf16 v[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          v[i] = (__bf16)((mask[L] >> (4 * mt + i)) & 1 ? h[i] : 0.0f);
          S.dz[L][(mt * 16 + 4 * q + i) * SP + sc] = v[i];
        }
        P[mt][0] = pack2(v[0], v[1]);
        P[mt][1] = pack2(v[2], v[3]);
      }
      if (L > 0) next_operand(P, b);
    }
    __syncthreads();
    // dW[in][out] of layer wv, one 32-sample set after the other
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      bf16x8 A[4];
#pragma unroll
      for (int mt = 0; mt < 4; mt++) A[mt] = load8(&S.in[wv][(mt * 16 + c16) * SP + ks * 32 + 8 * q]);
#pragma unroll
      for (int nt = 0; nt < 4; nt++) {
        if (nt >= NT) break;
        const bf16x8 B = load8(tz + (nt * 16 + c16) * SP + ks * 32 + 8 * q);
#pragma unroll
        for (int mt = 0; mt < 4; mt++) acc[mt][nt] = mma(A[mt], B, acc[mt][nt]);
      }
      if (l < nout) {
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const bf16x8 v = load8(tz + l * SP + ks * 32 + 8 * k);
#pragma unroll
          for (int j = 0; j < 8; j++) s += (float)v[j];
        }
        bacc += s;
      }
      if ((t0 + ks) % C == C - 1) {  // the slot is done
        if (per == 2) {
          store(acc, bacc, ch * 4 + (t0 + ks) / C);
        } else {
#pragma unroll
          for (int mt = 0; mt < 4; mt++)
#pragma unroll
            for (int nt = 0; nt < 4; nt++) g[mt][nt] += acc[mt][nt];
          bsum += bacc;
        }
#pragma unroll
        for (int mt = 0; mt < 4; mt++)
#pragma unroll
          for (int nt = 0; nt < 4; nt++) acc[mt][nt] = f32x4{0, 0, 0, 0};
        bacc = 0.0f;
      }
    }
    __syncthreads();  // the next pass reuses the tiles
  }
  if (per == 4) store(g, bsum, ch);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) lsum += __shfl_xor(lsum, off, 64);
  if (l == 0) S.red[wv] = lsum;
  __syncthreads();
  if (threadIdx.x == 0) loss_part[blockIdx.x] = (S.red[0] + S.red[1]) + (S.red[2] + S.red[3]);
}

// --------------------------------------------------------------- update --
// Gradient g = sum of the chunks' gradients in order (SLOTS: each the sum of its
// four slots in order), 64 loads in flight; ADAM then updates master/m/v
// (padded kernel layout) and refreshes the BF16 weight copies in both orientations
// and the FP32 biases.  Padding entries have zero gradient and stay zero.  The
// last block sums the loss partials, in FP64 as they are formed.
struct AdamArgs {
  float *master, *m1, *m2;
  float lr, b1, b2, eps, c1, c2;
};
template <bool ADAM, bool SLOTS>
__global__ __launch_bounds__(64) void k_mlp_update(const float *__restrict__ part, const double *__restrict__ loss_part,
                                                   int nchunk, int nloss, float *__restrict__ g,
                                                   std::conditional_t<ADAM, float, double> *__restrict__ loss,
                                                   AdamArgs a, Weights w) {
  if (blockIdx.x == gridDim.x - 1) {
    double s = 0.0;
    for (int b = threadIdx.x; b < nloss; b += 64) s += loss_part[b];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (threadIdx.x == 0) *loss = (std::conditional_t<ADAM, float, double>)s;
    return;
  }
  const int i = blockIdx.x * 64 + threadIdx.x;
  if (i >= GSIZE) return;
  constexpr int V = SLOTS ? 4 : 1, U = 64 / V;  // vectors per chunk, chunks per round
  float gi = 0.0f;
  auto chunk_sum = [&](const float *v) {
    if constexpr (SLOTS) return ((v[0] + v[1]) + v[2]) + v[3];
    else return v[0];
  };
  int c = 0;
  for (; c + U <= nchunk; c += U) {
    float v[64];
#pragma unroll
    for (int k = 0; k < 64; k++) v[k] = part[((size_t)c * V + k) * GSIZE + i];
#pragma unroll
    for (int k = 0; k < U; k++) gi += chunk_sum(v + k * V);
  }
  for (; c < nchunk; c++) {
    float v[V];
#pragma unroll
    for (int k = 0; k < V; k++) v[k] = part[((size_t)c * V + k) * GSIZE + i];
    gi += chunk_sum(v);
  }
  if constexpr (ADAM) {
    const float mi = a.b1 * a.m1[i] + (1.0f - a.b1) * gi;
    const float vi = a.b2 * a.m2[i] + (1.0f - a.b2) * gi * gi;
    a.m1[i] = mi;
    a.m2[i] = vi;
    const float p = a.master[i] - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
    a.master[i] = p;
    write_param(w, i, p);
  } else {
    g[i] = gi;
  }
}

// copies the padded FP32 master to the BF16 / bias arrays (after set_params)
__global__ __launch_bounds__(256) void k_mlp_refresh(const float *__restrict__ master, Weights w) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < GSIZE) write_param(w, i, master[i]);
}

}  // namespace mlp
}  // namespace chan

// ================================================================ C-ABI ==
#include <algorithm>
#include <cstring>
#include <vector>

#include "../../include/channel_closure.h"
#include "../../include/channel_hip.h"
#include "host_copy.hpp"

using namespace chan;
using namespace chan::mlp;

static_assert(NPARAM == CHAN_MLP_NPARAM, "canonical parameter count");

struct chan_mlp {
  int64_t cap = 0, n = 0;
  int dev = 0;                // device the model lives on
  int ncu = 256;              // its compute units
  hipStream_t st = nullptr;
  __bf16 *X = nullptr;        // [cap][64]
  float *T = nullptr;         // [cap][6]
  float *Xf = nullptr;        // [cap][46] host rows on their way in, made on first use
  float *Y = nullptr;         // [cap][6], at least [CHAN_MLP_NOALLOC_MAX][6]
  float *master = nullptr, *m1 = nullptr, *m2 = nullptr, *g = nullptr;  // [GSIZE]
  float *part = nullptr;      // gradient partials [gvec][GSIZE]
  double *lpart = nullptr;    // loss partials [GBLK], then the loss of chan_mlp_grad
  float *losses = nullptr;    // per training step
  __bf16 *woi = nullptr, *wio = nullptr;
  float *bias = nullptr;
  int64_t adam_t = 0;
  int losses_cap = 0;
  int gvec = 0;               // gradient partials
  HostStage stage;            // of rows on their way to and from the host
};

namespace {

// most chunks of a minibatch, and most partial vectors
constexpr int GBLK = 256;

#define MCHK(expr)                                                                                          \
  do {                                                                                                      \
    hipError_t e_ = (expr);                                                                                 \
    if (e_ != hipSuccess) return set_error((int)e_, "%s: %s", #expr, hipGetErrorString(e_));               \
  } while (0)

template <class T>
int mal(T **p, size_t n) {
  hipError_t e = hipMalloc((void **)p, n * sizeof(T) + 256);
  if (e != hipSuccess) return set_error((int)e, "hipMalloc of %zu bytes failed", n * sizeof(T));
  return 0;
}

Weights weights(chan_mlp *m) { return Weights{m->woi, m->wio, m->bias}; }

__global__ void k_to_bf16(const float *__restrict__ x, __bf16 *__restrict__ xb, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n * KP) return;
  const int64_t r = i / KP;
  const int c = (int)(i % KP);
  xb[i] = (__bf16)(c < IN ? x[r * IN + c] : 0.0f);
}

__global__ __launch_bounds__(256) void k_move_outputs(const float *__restrict__ a, float *__restrict__ b, int n) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) b[i] = a[i];
}

// Blocks of k_mlp_fwd: its waves keep the weights in registers, so each takes
// several tiles (two waves per SIMD are resident).
int fwd_blocks(const chan_mlp *m, int64_t n) {
  return (int)std::min<int64_t>(2 * (int64_t)m->ncu, std::max<int64_t>(1, ((n + 15) / 16 + 3) / 4));
}

template <class Src>
hipError_t launch_fwd(chan_mlp *m, const Src &src, int64_t n, float *Y, hipStream_t st) {
  hipLaunchKernelGGL((k_mlp_fwd<Src>), dim3(fwd_blocks(m, n)), dim3(256), 0, st, weights(m), src, (int)n, Y);
  return hipGetLastError();
}

// Gradient of the minibatch [first, first+count): partials, then their sum into
// m->g and the loss sum to lpart[GBLK] or, with `adam`, straight into the weights
// and *loss.
// Chunks are whole multiples of 128 samples, at most GBLK of them; up to GBLK / 4
// chunks are worked on slot by slot, by two blocks each.
int grad_pass(chan_mlp *m, int64_t first, int count, const AdamArgs *adam, float *loss) {
  const int wb = (int)std::min<int64_t>(GBLK, ((int64_t)count + 127) / 128);
  const int chunk = (int)((((int64_t)count + wb - 1) / wb + 127) / 128 * 128);
  const int nchunk = (count + chunk - 1) / chunk;
  const bool slots = nchunk <= GBLK / 4;
  const int nb = slots ? 2 * nchunk : nchunk;
  hipLaunchKernelGGL(k_mlp_grad, dim3(nb), dim3(256), sizeof(GradLds), m->st, weights(m), m->X + first * KP,
                     m->T + first * OUT, count, 1.0f / (6.0f * count), chunk, slots ? 2 : 4, m->part, m->lpart);
  MCHK(hipGetLastError());
  auto update = [&](auto kernel, auto *sum) {
    hipLaunchKernelGGL(kernel, dim3((GSIZE + 63) / 64 + 1), dim3(64), 0, m->st, m->part, m->lpart, nchunk, nb, m->g, sum,
                       adam ? *adam : AdamArgs{}, weights(m));
    return hipGetLastError();
  };
  if (adam)
    MCHK(slots ? update(k_mlp_update<true, true>, loss) : update(k_mlp_update<true, false>, loss));
  else
    MCHK(slots ? update(k_mlp_update<false, true>, m->lpart + GBLK) : update(k_mlp_update<false, false>, m->lpart + GBLK));
  return 0;
}

// The stream's end, whatever failed before: until then a transfer may still read the
// caller's rows.
hipError_t settle(chan_mlp *m, hipError_t e) {
  const hipError_t end = hipStreamSynchronize(m->st);
  return e != hipSuccess ? e : end;
}

int row_workspace(chan_mlp *m) {
  int rc;
  if (!m->Xf && (rc = mal(&m->Xf, (size_t)m->cap * IN))) return rc;
  return 0;
}

}  // namespace

hipError_t chan::mlp::forward_gradients(chan_mlp *m, const LesSource &s, float *Y, hipStream_t st) {
  if (s.n < 1 || s.n > ((int64_t)1 << 31) / KP) return hipErrorInvalidValue;
  const int nb = (int)std::min<int64_t>(2 * (int64_t)m->ncu, ((int64_t)s.n + 255) / 256);
  hipLaunchKernelGGL(k_mlp_fwd_les, dim3(nb), dim3(256), 0, st, weights(m), s, s.norm, s.yplus, Y);
  return hipGetLastError();
}

extern "C" {

int chan_mlp_create(int64_t capacity, chan_mlp **out) {
  if (!out || capacity < 1 || capacity > ((int64_t)1 << 31) / KP) return set_error(CHAN_E_ARG, "bad capacity");
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return set_error(CHAN_E_NODEV, "no HIP device");
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return set_error(CHAN_E_NODEV, "no current HIP device");
  int rc = 0;
  chan_mlp *m = new chan_mlp();
  m->cap = capacity;
  m->dev = dev;
  if (hipDeviceGetAttribute(&m->ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || m->ncu < 1) m->ncu = 256;
  // gradient vectors: four slots of each of GBLK / 4 chunks, or GBLK chunks
  m->gvec = (int)std::min<int64_t>(GBLK, (capacity + 127) / 128 * 4);
  auto bail = [&](int code) {
    chan_mlp_destroy(m);
    return code;
  };
  if (hipStreamCreate(&m->st) != hipSuccess) return bail(set_error(CHAN_E_STATE, "hipStreamCreate failed"));
  const size_t c = (size_t)capacity;
  if ((rc = mal(&m->X, c * KP)) || (rc = mal(&m->T, c * OUT)) || (rc = mal(&m->Y, std::max(c, (size_t)CHAN_MLP_NOALLOC_MAX) * OUT)) ||
      (rc = mal(&m->master, GSIZE)) || (rc = mal(&m->m1, GSIZE)) || (rc = mal(&m->m2, GSIZE)) ||
      (rc = mal(&m->g, GSIZE)) || (rc = mal(&m->part, (size_t)m->gvec * GSIZE)) ||
      (rc = mal(&m->lpart, (size_t)GBLK + 1)) ||
      (rc = mal(&m->woi, WSIZE)) || (rc = mal(&m->wio, WSIZE)) || (rc = mal(&m->bias, BSIZE)))
    return bail(rc);
  if (hipMemset(m->master, 0, sizeof(float) * GSIZE) != hipSuccess ||
      hipMemset(m->m1, 0, sizeof(float) * GSIZE) != hipSuccess || hipMemset(m->m2, 0, sizeof(float) * GSIZE) != hipSuccess ||
      hipMemset(m->woi, 0, sizeof(__bf16) * WSIZE) != hipSuccess || hipMemset(m->wio, 0, sizeof(__bf16) * WSIZE) != hipSuccess ||
      hipMemset(m->bias, 0, sizeof(float) * BSIZE) != hipSuccess)
    return bail(set_error(CHAN_E_STATE, "hipMemset failed"));
  *out = m;
  return 0;
}

int chan_mlp_destroy(chan_mlp *m) {
  if (!m) return 0;
  if (m->st) hipStreamSynchronize(m->st);
  m->stage.free();
  void *bufs[] = {m->X, m->T, m->Xf, m->Y, m->master, m->m1, m->m2, m->g, m->part, m->lpart,
                  m->losses, m->woi, m->wio, m->bias};
  for (void *b : bufs)
    if (b) hipFree(b);
  if (m->st) hipStreamDestroy(m->st);
  delete m;
  return 0;
}

int chan_mlp_set_params(chan_mlp *m, const float *params) {
  if (!m || !params) return set_error(CHAN_E_ARG, "null argument");
  std::vector<float> pad(GSIZE, 0.0f);
  for (int c = 0; c < NPARAM; c++) pad[canon_to_padded(c)] = params[c];
  hipError_t e = hipMemcpyAsync(m->master, pad.data(), sizeof(float) * GSIZE, hipMemcpyHostToDevice, m->st);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_mlp_refresh, dim3((GSIZE + 255) / 256), dim3(256), 0, m->st, m->master, weights(m));
    e = hipGetLastError();
  }
  MCHK(settle(m, e));
  return 0;
}

int chan_mlp_get_params(chan_mlp *m, float *params) {
  if (!m || !params) return set_error(CHAN_E_ARG, "null argument");
  std::vector<float> pad(GSIZE);
  MCHK(hipMemcpyAsync(pad.data(), m->master, sizeof(float) * GSIZE, hipMemcpyDeviceToHost, m->st));
  MCHK(hipStreamSynchronize(m->st));
  for (int c = 0; c < NPARAM; c++) params[c] = pad[canon_to_padded(c)];
  return 0;
}

int chan_mlp_set_data(chan_mlp *m, const float *X, const float *T, int64_t n) {
  if (!m || !X || !T || n < 1 || n > m->cap) return set_error(CHAN_E_ARG, "bad argument");
  int rc;
  if ((rc = row_workspace(m))) return rc;
  hipError_t e = copy_to_device(m->stage, m->Xf, X, sizeof(float) * n * IN, m->st);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_to_bf16, dim3((unsigned)((n * KP + 255) / 256)), dim3(256), 0, m->st, m->Xf, m->X, n);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = copy_to_device(m->stage, m->T, T, sizeof(float) * n * OUT, m->st);
  if (e == hipSuccess) e = hipMemsetAsync(m->m1, 0, sizeof(float) * GSIZE, m->st);
  if (e == hipSuccess) e = hipMemsetAsync(m->m2, 0, sizeof(float) * GSIZE, m->st);
  e = settle(m, e);
  if (e != hipSuccess) return set_error((int)e, "set_data: %s", hipGetErrorString(e));
  m->n = n;
  m->adam_t = 0;
  return 0;
}

int chan_mlp_forward(chan_mlp *m, const float *X, int64_t n, float *Y) {
  if (!m || !X || !Y || n < 1 || n > m->cap) return set_error(CHAN_E_ARG, "bad argument");
  int rc;
  if ((rc = row_workspace(m))) return rc;
  hipError_t e = copy_to_device(m->stage, m->Xf, X, sizeof(float) * n * IN, m->st);
  if (e == hipSuccess) e = launch_fwd(m, FromFloat{m->Xf}, n, m->Y, m->st);
  if (e == hipSuccess) e = copy_to_host(m->stage, Y, m->Y, sizeof(float) * n * OUT, m->st);
  if (e != hipSuccess) return set_error((int)settle(m, e), "forward: %s", hipGetErrorString(e));
  return 0;
}

int chan_mlp_forward_noalloc(chan_mlp *m, const float *dX, int64_t n, float *dY) {
  if (!m || !dX || !dY || n < 1) return set_error(CHAN_E_ARG, "bad argument");
  if (n > CHAN_MLP_NOALLOC_MAX)
    return set_error(CHAN_E_ARG, "chan_mlp_forward_noalloc: %lld rows exceed its limit of %d rows; split the call",
                     (long long)n, CHAN_MLP_NOALLOC_MAX);
  int dev = -1;
  MCHK(hipGetDevice(&dev));
  if (dev != m->dev) return set_error(CHAN_E_STATE, "chan_mlp_forward_noalloc: device %d is current, the model lives on %d", dev, m->dev);
  // the same kernel and launch shape as chan_mlp_forward.  Its waves store outputs
  // while others still read rows: buffers that overlap go through the model's own
  // output rows.
  const uintptr_t x = (uintptr_t)dX, y = (uintptr_t)dY;
  const bool overlap = x < y + (size_t)n * OUT * sizeof(float) && y < x + (size_t)n * IN * sizeof(float);
  MCHK(launch_fwd(m, FromFloat{dX}, n, overlap ? m->Y : dY, m->st));
  if (overlap) {
    hipLaunchKernelGGL(k_move_outputs, dim3((unsigned)std::min<int64_t>(256, (n * OUT + 255) / 256)), dim3(256), 0, m->st,
                       m->Y, dY, (int)(n * OUT));
    MCHK(hipGetLastError());
  }
  MCHK(hipStreamSynchronize(m->st));
  return 0;
}

int chan_mlp_grad(chan_mlp *m, int64_t first, int64_t count, float *grad, double *loss) {
  if (!m || !grad || !loss || first < 0 || count < 1 || first + count > m->n) return set_error(CHAN_E_ARG, "bad argument");
  int rc;
  if ((rc = grad_pass(m, first, (int)count, nullptr, nullptr))) return rc;
  std::vector<float> pad(GSIZE);
  double lsum = 0.0;
  MCHK(hipMemcpyAsync(pad.data(), m->g, sizeof(float) * GSIZE, hipMemcpyDeviceToHost, m->st));
  MCHK(hipMemcpyAsync(&lsum, m->lpart + GBLK, sizeof lsum, hipMemcpyDeviceToHost, m->st));
  MCHK(hipStreamSynchronize(m->st));
  for (int c = 0; c < NPARAM; c++) grad[c] = pad[canon_to_padded(c)];
  *loss = lsum / (6.0 * (double)count);
  return 0;
}

int chan_mlp_train(chan_mlp *m, int32_t steps, int32_t batch, float lr, float *losses, double *ms_per_step) {
  if (!m || steps < 1 || batch < 16 || batch > m->n || !(lr > 0)) return set_error(CHAN_E_ARG, "bad argument");
  if (m->losses_cap < steps) {
    if (m->losses) hipFree(m->losses);
    m->losses = nullptr;
    int rc;
    if ((rc = mal(&m->losses, (size_t)steps))) return rc;
    m->losses_cap = steps;
  }
  hipEvent_t e0, e1;
  MCHK(hipEventCreate(&e0));
  MCHK(hipEventCreate(&e1));
  MCHK(hipEventRecord(e0, m->st));
  int64_t off = 0;
  for (int s = 0; s < steps; s++) {
    if (off + batch > m->n) off = 0;
    m->adam_t++;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - (float)std::pow((double)b1, (double)m->adam_t);
    const float c2 = 1.0f - (float)std::pow((double)b2, (double)m->adam_t);
    const AdamArgs adam = {m->master, m->m1, m->m2, lr, b1, b2, 1e-8f, c1, c2};
    int rc;
    if ((rc = grad_pass(m, off, batch, &adam, m->losses + s))) return rc;
    off += batch;
  }
  MCHK(hipEventRecord(e1, m->st));
  MCHK(hipEventSynchronize(e1));
  float ms = 0;
  MCHK(hipEventElapsedTime(&ms, e0, e1));
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  if (ms_per_step) *ms_per_step = ms / steps;
  if (losses) {
    std::vector<float> l(steps);
    MCHK(hipMemcpy(l.data(), m->losses, sizeof(float) * steps, hipMemcpyDeviceToHost));
    for (int s = 0; s < steps; s++) losses[s] = l[s] / (6.0f * batch);
  }
  return 0;
}

int chan_mlp_bench_forward(chan_mlp *m, int32_t reps, double *ms) {
  if (!m || reps < 1 || !ms || m->n < 1) return set_error(CHAN_E_ARG, "bad argument");
  hipEvent_t e0, e1;
  MCHK(hipEventCreate(&e0));
  MCHK(hipEventCreate(&e1));
  const int n = (int)m->n;
  MCHK(launch_fwd(m, FromBf16{m->X}, n, m->Y, m->st));
  MCHK(hipEventRecord(e0, m->st));
  for (int r = 0; r < reps; r++) MCHK(launch_fwd(m, FromBf16{m->X}, n, m->Y, m->st));
  MCHK(hipEventRecord(e1, m->st));
  MCHK(hipEventSynchronize(e1));
  float t = 0;
  MCHK(hipEventElapsedTime(&t, e0, e1));
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  *ms = t / reps;
  return 0;
}

}  // extern "C"
