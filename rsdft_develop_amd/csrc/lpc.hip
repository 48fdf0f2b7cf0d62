// lpc.hip -- learned CG preconditioner: a 3-layer 3x3x3 convolution net on
// the periodic grid that maps a band residual g and the cell's normalised
// local potential v to a correction P g (replacing precond_hprsdft,
// cgpc_hprsdft_module.f90:133-361, which has no learned counterpart in the
// reference):
//
//   s = rms(g); x = [g/s, v]
//   a1 = relu(W1 * x + b1)   (2 -> 16)
//   a2 = relu(W2 * a1 + b2)  (16 -> 16)
//   y  = W3 * a2 + b3        (16 -> 1)
//   P g = s y                (scale-equivariant: P(c g) = c P g)
//
// Storage: weights and activations in bfloat16, channel-last
// (act[sample][point][channel]); every product on MFMA
// (v_mfma_f32_16x16x16bf16_1k) with FP32 accumulation.  A convolution is
// D[co][p] = sum_k W[co][k] X[k][p] over k = tap * CIN + ci, tap = d3*9 +
// d2*3 + d1, with X[k][p] = in[point p shifted by (d - 1), periodic][ci];
// the weight matrix is the MFMA A operand and 16 grid points form the B
// operand, so a lane's output is 4 consecutive channels of one point.
// The input gradient of a layer is the same convolution with the adjoint
// weights W'[ci][tap' * COUT + co] = W[co][ci][26 - tap'].
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "lpc.hpp"
#include "solver.hpp"

namespace rsg {
namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;  // waves per workgroup in the convolution kernels

__host__ __device__ inline uint16_t f2bf(float f) {
  uint32_t u;
  __builtin_memcpy(&u, &f, 4);
  if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x7fffffu)) return uint16_t((u >> 16) | 0x40);  // NaN stays NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return uint16_t(u >> 16);
}
__host__ __device__ inline float bf2f(uint16_t h) {
  uint32_t u = uint32_t(h) << 16;
  float f;
  __builtin_memcpy(&f, &u, 4);
  return f;
}

struct Grid3 {
  int n1, n2, n3;
};

__device__ inline bf16x4 as_bf16x4(uint2 w) {
  bf16x4 v;
  v[0] = short(w.x & 0xffff);
  v[1] = short(w.x >> 16);
  v[2] = short(w.y & 0xffff);
  v[3] = short(w.y >> 16);
  return v;
}

// i + d - 1 on an axis of n points, periodic
__device__ inline int tap_wrap(int i, int d, int n) {
  const int j = i + d - 1;
  return j < 0 ? j + n : (j >= n ? j - n : j);
}

enum ConvMode { kReluOut = 0, kFinalOut = 1, kMaskedGrad = 2 };

// One convolution layer for nsamp samples.  Modes:
//  kReluOut:   out_bf[p][co] = bf16(relu(D + bias))            (16 outputs)
//  kFinalOut:  y = D[0] + bias[0]; yout[p] = y (FP32 if non-null);
//              pg[p] = s y  (the preconditioned residual, type T)
//  kMaskedGrad: out_bf[p][co] = bf16(D * (mask[p][co] > 0))    (16 outputs)
//
// A wave owns 16 consecutive points of an xy-plane of one sample and walks
// a run of z-planes.  The in-plane offsets of its neighbours are the same
// in every plane, so they are formed once.  With 16 input channels (a K
// chunk of 16 is one tap) the nine fragments of a plane serve the three
// output planes it touches: it is the d3 = 2 tap plane of the output below,
// d3 = 1 of its own and d3 = 0 of the output above, each with its own
// accumulators.  9 loads feed 27 products, where a gather of each tap took
// 27 loads and their address arithmetic.  Three accumulator chains per
// output (taps c mod 3, that is d1): one chain's latency would bound the
// tile.  With one or two input channels a lane's K slots are different
// taps, loaded for each output plane.  Bound: matrix-core issue.  A layer of
// 16 channels issues 27 K = 16 products per 16 points, 0.83 TFLOP for 160
// bands of 72^3, in 1.80 ms (16 outputs) and 1.44 ms (one output in a tile
// of 16): 458 and 572 TFLOP/s.  A large bf16 product reaches 1163 with the
// K = 32 form, whose instructions do twice the work.
// The three layers of 160 bands of 72^3 points, FP32 in and out: 4.3 ms,
// 12.4 with a gather per tap; same values.
template <int CIN, int KP, int MODE, typename T>
__global__ __launch_bounds__(64 * kWaves) void k_conv(Grid3 g, int64_t N, int zlen, int nzr, int ntg,
                                                      const uint16_t *__restrict__ in, int64_t in_stride,
                                                      const uint16_t *__restrict__ wbf,
                                                      const float *__restrict__ bias, uint16_t *__restrict__ out_bf,
                                                      const uint16_t *__restrict__ mask, float *__restrict__ yout,
                                                      T *__restrict__ pg, int64_t ldg,
                                                      const float *__restrict__ sval) {
  constexpr int NC = KP / 16;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lq = lane >> 4, lr = lane & 15;
  // logical block: tile group fastest, then z-run, then sample; each XCD
  // takes one contiguous range, so neighbouring tiles share an L2
  const unsigned nblk = gridDim.x, xc = blockIdx.x % 8;
  const unsigned lb = xc * (nblk / 8) + min(xc, nblk % 8) + blockIdx.x / 8;
  const int tg = int(lb % unsigned(ntg)), zr = int((lb / unsigned(ntg)) % unsigned(nzr));
  const int smp = int(lb / unsigned(ntg * nzr));
  const int n12 = g.n1 * g.n2, j0 = (tg * kWaves + wave) * 16;
  if (j0 >= n12) return;  // whole wave; no barriers in this kernel
  const uint16_t *__restrict__ src = in + int64_t(smp) * in_stride;
  const int j = min(j0 + lr, n12 - 1), x = j % g.n1, y = j / g.n1;
  const bool ok = j0 + lr < n12;
  const int z0 = zr * zlen, z1 = min(z0 + zlen, g.n3);
  // A fragments: W[co = lr][k = 16c + 4 lq + i]
  bf16x4 a[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) a[c] = as_bf16x4(*reinterpret_cast<const uint2 *>(wbf + lr * KP + 16 * c + 4 * lq));
  float bs[4] = {0.f, 0.f, 0.f, 0.f};
  if constexpr (MODE == kReluOut) {
#pragma unroll
    for (int i = 0; i < 4; ++i) bs[i] = bias[4 * lq + i];
  }
  const float b0 = MODE == kFinalOut ? bias[0] : 0.f;
  auto finish = [&](int z, const f32x4 (&acc3)[3]) {
    const f32x4 acc = (acc3[0] + acc3[1]) + acc3[2];
    const int64_t p = int64_t(z) * n12 + j;
    if constexpr (MODE == kReluOut || MODE == kMaskedGrad) {
      const int64_t o = int64_t(smp) * N * 16 + p * 16 + 4 * lq;
      uint16_t h[4];
      bf16x4 m{};
      if constexpr (MODE == kMaskedGrad) m = as_bf16x4(*reinterpret_cast<const uint2 *>(mask + o));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v = acc[i];
        if constexpr (MODE == kReluOut) {
          v += bs[i];
          v = v > 0.f ? v : 0.f;
        } else {
          v = bf2f(uint16_t(m[i])) > 0.f ? v : 0.f;
        }
        h[i] = f2bf(v);
      }
      if (ok) {
        uint2 w;
        w.x = uint32_t(h[0]) | (uint32_t(h[1]) << 16);
        w.y = uint32_t(h[2]) | (uint32_t(h[3]) << 16);
        *reinterpret_cast<uint2 *>(out_bf + o) = w;
      }
    } else {
      // row co = 0 lives in acc[0] of lanes 0..15
      if (lq == 0 && ok) {
        const float yv = acc[0] + b0;
        if (yout) yout[int64_t(smp) * N + p] = yv;
        if (pg) pg[int64_t(smp) * ldg + p] = T(double(sval[smp]) * double(yv));
      }
    }
  };
  if constexpr (CIN == 16) {
    // points of the plane; the channel factor goes into the 64-bit address
    // (a plane of 2^27 points passes 2^31 channels)
    unsigned ofs[9];
#pragma unroll
    for (int t = 0; t < 9; ++t) ofs[t] = unsigned(tap_wrap(x, t % 3, g.n1) + g.n1 * tap_wrap(y, t / 3, g.n2));
    const int64_t pstr = int64_t(n12) * 16;
    f32x4 acc[3][3];  // [output plane mod 3][chain]
    uint2 nf[9];
    int zn = z0 == 0 ? g.n3 - 1 : z0 - 1;  // input plane to fetch
    auto fetch = [&]() {
      const uint16_t *sp = src + zn * pstr + 4 * lq;
#pragma unroll
      for (int t = 0; t < 9; ++t) nf[t] = *reinterpret_cast<const uint2 *>(sp + size_t(ofs[t]) * 16);
      zn = zn + 1 == g.n3 ? 0 : zn + 1;
    };
    fetch();
    // step s: input plane z0 - 1 + s; U = s mod 3 is the slot of output s (plane z0 + s)
    auto step = [&](int s, auto uc) {
      constexpr int U = decltype(uc)::value, Um1 = (U + 2) % 3, Um2 = (U + 1) % 3;
      uint2 f[9];
#pragma unroll
      for (int t = 0; t < 9; ++t) f[t] = nf[t];
      if (s + 1 < z1 - z0 + 2) fetch();
#pragma unroll
      for (int d = 0; d < 3; ++d) acc[U][d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        const bf16x4 b = as_bf16x4(f[t]);
        acc[U][t % 3] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[t], b, acc[U][t % 3], 0, 0, 0);
        acc[Um1][t % 3] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[9 + t], b, acc[Um1][t % 3], 0, 0, 0);
        acc[Um2][t % 3] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[18 + t], b, acc[Um2][t % 3], 0, 0, 0);
      }
      if (s >= 2) finish(z0 + s - 2, acc[Um2]);  // outputs s - 2 >= 0 are complete
    };
#pragma unroll
    for (int u = 0; u < 3; ++u)
#pragma unroll
      for (int d = 0; d < 3; ++d) acc[u][d] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int ns = z1 - z0 + 2;
    for (int s = 0; s < ns; s += 3) {
      step(s, std::integral_constant<int, 0>{});
      if (s + 1 < ns) step(s + 1, std::integral_constant<int, 1>{});
      if (s + 2 < ns) step(s + 2, std::integral_constant<int, 2>{});
    }
  } else {
    // K slot k = 16 c + 4 lq + i is channel k % CIN of tap k / CIN: the
    // lane's taps, their in-plane offsets and planes
    constexpr int NT = NC * 4 / CIN;
    unsigned ofs[NT];
    int dz[NT];
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const int t = (16 * (u / (4 / CIN)) + 4 * lq) / CIN + u % (4 / CIN), tc = min(t, 26);
      dz[u] = t < 27 ? tc / 9 : 3;  // 3: no tap
      ofs[u] = unsigned(tap_wrap(x, tc % 3, g.n1) + g.n1 * tap_wrap(y, (tc / 3) % 3, g.n2));
    }
    const int64_t pstr = int64_t(n12) * CIN;
    for (int z = z0; z < z1; ++z) {
      const uint16_t *s0 = src + tap_wrap(z, 0, g.n3) * pstr, *s1 = src + z * pstr, *s2 = src + tap_wrap(z, 2, g.n3) * pstr;
      f32x4 acc3[3] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      uint32_t w[NT];
#pragma unroll
      for (int u = 0; u < NT; ++u) {
        const uint16_t *p = (dz[u] == 0 ? s0 : (dz[u] == 2 ? s2 : s1)) + size_t(ofs[u]) * CIN;
        if constexpr (CIN == 2)
          w[u] = *reinterpret_cast<const uint32_t *>(p);
        else
          w[u] = *p;
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        bf16x4 b;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int u = (4 / CIN) * c + i / CIN;
          const uint32_t v = dz[u] == 3 ? 0u : (CIN == 2 && (i & 1) ? w[u] >> 16 : w[u]);
          b[i] = short(v & 0xffff);
        }
        acc3[c % 3] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[c], b, acc3[c % 3], 0, 0, 0);
      }
      finish(z, acc3);
    }
  }
}

// x[smp][p] = (bf16(g/s), bf16(v))
template <typename T>
__global__ void k_prep(const T *__restrict__ gsrc, int64_t ldg, const float *__restrict__ v,
                       const float *__restrict__ sval, int64_t N, uint16_t *__restrict__ x) {
  const int smp = blockIdx.y;
  const int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (p >= N) return;
  const float s = sval[smp];
  const float g = float(double(gsrc[int64_t(smp) * ldg + p]) / double(s));
  const uint32_t w = uint32_t(f2bf(g)) | (uint32_t(f2bf(v[p])) << 16);
  *reinterpret_cast<uint32_t *>(x + (int64_t(smp) * N + p) * 2) = w;
}

// s = sqrt(<g,g>/N) per sample, with a floor that keeps 0/0 out
__global__ void k_rms(const double *__restrict__ gg, int nsamp, int64_t N, float *__restrict__ s) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nsamp) s[i] = float(fmax(sqrt(gg[i] / double(N)), 1e-30));
}

// Loss of a batch: r = y - kappa t / s, L += sum r^2 / (N nsamp);
// dy = 2 r / (N nsamp) stored as bf16 for the backward convolutions.
__global__ __launch_bounds__(256) void k_loss(const float *__restrict__ tgt, const float *__restrict__ y,
                                              const float *__restrict__ sval, float kappa, int64_t N,
                                              double inv_count, uint16_t *__restrict__ dy,
                                              double *__restrict__ lsum) {
  __shared__ double red[4];
  const int smp = blockIdx.y;
  const int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  double r2 = 0.0;
  if (p < N) {
    const int64_t o = int64_t(smp) * N + p;
    const float r = y[o] - kappa * tgt[o] / sval[smp];
    r2 = double(r) * r;
    dy[o] = f2bf(float(2.0 * inv_count * r));
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) r2 += __shfl_xor(r2, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = r2;
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(lsum, (red[0] + red[1] + red[2] + red[3]) * inv_count);
}

// Quad layout of a channel-last field for products that contract over the
// points: out[row][quad][channel][4 points], a row being one x-line of one
// sample.  Quad q holds the points x = 4 (q - 1) .. 4 (q - 1) + 3, so each
// line has a quad in front of it; with wrap the points x = -1 and x = n1
// are the periodic copies, everything else outside 0..n1-1 is zero.
template <int C>
__global__ __launch_bounds__(256) void k_quads(const uint16_t *__restrict__ in, int64_t nrow, int n1, int nq, int wrap,
                                               uint16_t *__restrict__ out) {
  const int64_t t = (int64_t(blockIdx.y) * gridDim.x + blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= nrow * nq * C) return;
  const int c = int(t % C), q = int((t / C) % nq);
  const int64_t row = t / (int64_t(C) * nq);
  uint16_t v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    int x = 4 * (q - 1) + i;
    if (wrap && x == -1) x = n1 - 1;
    else if (wrap && x == n1) x = 0;
    v[i] = x >= 0 && x < n1 ? in[(row * n1 + x) * C + c] : uint16_t(0);
  }
  uint2 w;
  w.x = uint32_t(v[0]) | (uint32_t(v[1]) << 16);
  w.y = uint32_t(v[2]) | (uint32_t(v[3]) << 16);
  *reinterpret_cast<uint2 *>(out + 4 * t) = w;
}

// dW[co][k] += sum_p dz[p][co] X[k][p], k = tap * CIN + ci, on MFMA with
// co x 16-k-chunk outputs and 16 points of an x-line per product.  Both
// operands hold four consecutive points of one channel per lane, so they
// are read from the quad layout, 512 contiguous bytes a wave; the taps with
// d1 = -1 and +1 shift the quad by one point with the quad beside it.  (A
// gather of single channels from the channel-last fields took 2-byte loads,
// 108 of them per lane and 16 points: 920 us against 75 us here for 16
// samples of 36^3 points.)  Lines past n1 are zero in dz.  A wave takes
// every (4 blocks)-th line; a block adds its four waves in order into part.
template <int CIN, int KP, int COUT>
__global__ __launch_bounds__(256) void k_conv_dw(Grid3 g, int nsamp, const uint16_t *__restrict__ xq,
                                                 const uint16_t *__restrict__ dq, int nq, float *__restrict__ part) {
  constexpr int NC = KP / 16;
  __shared__ float red[16 * KP];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lq = lane >> 4, lr = lane & 15;
  f32x4 acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int n23 = g.n2 * g.n3, nrow = n23 * nsamp, nch = (g.n1 + 15) / 16;
  for (int row = blockIdx.x * 4 + wave; row < nrow; row += 4 * gridDim.x) {
    const int smp = row / n23, zy = row - smp * n23, z = zy / g.n2, y = zy - z * g.n2;
    int rz[3], ry[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int zz = z + d - 1, yy = y + d - 1;
      rz[d] = smp * n23 + g.n2 * (zz < 0 ? zz + g.n3 : (zz >= g.n3 ? zz - g.n3 : zz));
      ry[d] = yy < 0 ? yy + g.n2 : (yy >= g.n2 ? yy - g.n2 : yy);
    }
    for (int ch = 0; ch < nch; ++ch) {
      const int qa = 1 + 4 * ch + lq;
      bf16x4 av = {0, 0, 0, 0};
      if (lr < COUT) av = as_bf16x4(*reinterpret_cast<const uint2 *>(dq + ((int64_t(row) * nq + qa) * COUT + lr) * 4));
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        // CIN = 16: the chunk is one tap, the same for every lane
        const int k = 16 * c + lr, tap = CIN == 16 ? c : min(k / CIN, 26), ci = CIN == 16 ? lr : k % CIN;
        const int d3 = tap / 9, d2 = (tap / 3) % 3, d1 = tap % 3;
        const int64_t r = (d3 == 0 ? rz[0] : (d3 == 1 ? rz[1] : rz[2])) + (d2 == 0 ? ry[0] : (d2 == 1 ? ry[1] : ry[2]));
        const uint16_t *p = xq + ((r * nq + qa) * CIN + ci) * 4;
        const uint2 w = *reinterpret_cast<const uint2 *>(p);
        // the point before the quad, or the one after it (the middle tap reads its own quad again)
        const uint32_t o = p[d1 == 0 ? 3 - 4 * CIN : (d1 == 2 ? 4 * CIN : 0)];
        uint2 v = w;
        if (d1 == 0) {
          v.x = o | (w.x << 16);
          v.y = (w.x >> 16) | (w.y << 16);
        } else if (d1 == 2) {
          v.x = (w.x >> 16) | (w.y << 16);
          v.y = (w.y >> 16) | (o << 16);
        }
        if (CIN != 16 && k / CIN > 26) v.x = v.y = 0;
        acc[c] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, as_bf16x4(v), acc[c], 0, 0, 0);
      }
    }
  }
  // D[co = 4 lq + i][k = 16c + lr]
  for (int w = 0; w < 4; ++w) {
    if (wave == w) {
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float &o = red[(4 * lq + i) * KP + 16 * c + lr];
          o = w == 0 ? acc[c][i] : o + acc[c][i];
        }
    }
    __syncthreads();
  }
  for (int i = threadIdx.x; i < 16 * KP; i += blockDim.x) part[int64_t(blockIdx.x) * 16 * KP + i] = red[i];
}

// out[i] = sum over nblk partial rows of len values: 64 columns a block,
// each of its 16 waves every 16th row, the waves added in order
__global__ __launch_bounds__(1024) void k_sum_parts(const float *__restrict__ part, int nblk, int len,
                                                    float *__restrict__ out) {
  __shared__ double red[16][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = blockIdx.x * 64 + lane;
  double s = 0.0;
  if (i < len)
    for (int b = wave; b < nblk; b += 16) s += part[int64_t(b) * len + i];
  red[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && i < len) {
    for (int w = 1; w < 16; ++w) s += red[w][lane];
    out[i] = float(s);
  }
}

// bias gradient: per block sum_p dz[p][co] (COUT channels, bf16) into part[block][COUT].  A
// thread reads eight channels (16 bytes) of a point at a time, or eight
// points where COUT is 1, neighbouring threads neighbouring words; the
// last words of a COUT = 1 field may hold fewer than eight points.
template <int COUT>
__global__ __launch_bounds__(256) void k_bias_grad(const uint16_t *__restrict__ dz, int64_t total,
                                                   float *__restrict__ part) {
  constexpr int H = COUT == 16 ? 2 : 1;  // words per point group
  __shared__ float red[4][16];
  float acc[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) acc[c] = 0.f;
  const int64_t nval = total * COUT, nword = nval / 8;
  for (int64_t q = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; q < nword; q += int64_t(gridDim.x) * blockDim.x) {
    const uint4 w = *reinterpret_cast<const uint4 *>(dz + 8 * q);
    const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      acc[2 * c] += bf2f(uint16_t(u[c] & 0xffff));
      acc[2 * c + 1] += bf2f(uint16_t(u[c] >> 16));
    }
  }
  if (COUT == 1 && blockIdx.x == 0 && threadIdx.x == 0)
    for (int64_t q = 8 * nword; q < nval; ++q) acc[0] += bf2f(dz[q]);
  if (COUT == 1) {
#pragma unroll
    for (int c = 1; c < 8; ++c) acc[0] += acc[c];
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int c = 0; c < (COUT == 1 ? 1 : 8); ++c) {
    float v = acc[c];
#pragma unroll
    for (int off = 32; off >= H; off >>= 1) v += __shfl_xor(v, off, 64);
    if (lane < H) red[wave][8 * lane + c] = v;  // lane parity: channels 0..7 or 8..15
  }
  __syncthreads();
  if (threadIdx.x < COUT)
    part[int64_t(blockIdx.x) * COUT + threadIdx.x] =
        (red[0][threadIdx.x] + red[1][threadIdx.x]) + (red[2][threadIdx.x] + red[3][threadIdx.x]);
}

// Adam on the FP32 master parameters
__global__ void k_adam(float *__restrict__ w, const float *__restrict__ gr, float *__restrict__ m,
                       float *__restrict__ v, int n, float lr, float b1, float b2, float eps, float c1,
                       float c2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = gr[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

}  // namespace

// ------------------------------------------------------------ host side

// Parameter vector layout (FP32 master, reference order):
//   W1[16][2][27] | b1[16] | W2[16][16][27] | b2[16] | W3[1][16][27] | b3[1]
// with W[co][ci][tap], tap = d3*9 + d2*3 + d1.
int lpc_param_count() { return 16 * 2 * 27 + 16 + 16 * 16 * 27 + 16 + 16 * 27 + 1; }

namespace {

constexpr int KP1 = 64, KP2 = 432, KP3 = 432, KP3T = 32;
constexpr int OFF_W1 = 0, OFF_B1 = 864, OFF_W2 = 880, OFF_B2 = 7792, OFF_W3 = 7808, OFF_B3 = 8240;

// bf16 weight matrices for the kernels, from the FP32 master vector
void pack_weights(const std::vector<float> &p, std::vector<uint16_t> &w) {
  w.assign(size_t(16) * (KP1 + KP2 + KP3 + KP2 + KP3T), 0);
  uint16_t *w1 = w.data(), *w2 = w1 + 16 * KP1, *w3 = w2 + 16 * KP2, *w2t = w3 + 16 * KP3, *w3t = w2t + 16 * KP2;
  for (int co = 0; co < 16; ++co)
    for (int ci = 0; ci < 2; ++ci)
      for (int t = 0; t < 27; ++t) w1[co * KP1 + t * 2 + ci] = f2bf(p[OFF_W1 + (co * 2 + ci) * 27 + t]);
  for (int co = 0; co < 16; ++co)
    for (int ci = 0; ci < 16; ++ci)
      for (int t = 0; t < 27; ++t) {
        const uint16_t h = f2bf(p[OFF_W2 + (co * 16 + ci) * 27 + t]);
        w2[co * KP2 + t * 16 + ci] = h;
        w2t[ci * KP2 + (26 - t) * 16 + co] = h;  // adjoint: rows ci, flipped taps
      }
  for (int ci = 0; ci < 16; ++ci)
    for (int t = 0; t < 27; ++t) {
      const uint16_t h = f2bf(p[OFF_W3 + ci * 27 + t]);
      w3[0 * KP3 + t * 16 + ci] = h;  // row 0 only
      w3t[ci * KP3T + (26 - t)] = h;  // adjoint: 1 input channel
    }
}

}  // namespace

LpcState::~LpcState() { release(); }

void LpcState::release() {
  for (DevBuf *b : {&wbf, &bias, &vnorm, &x0, &a1, &a2, &y, &dyb, &dz1, &dz2, &sval, &gg, &part, &grad, &master, &mom1,
                    &mom2, &lsum, &diag, &tbuf, &xq, &dq})
    b->release();
}

int lpc_set_params(rsg_ctx *ctx, const float *params) {
  LpcState &L = ctx->lpc;
  const int n = lpc_param_count();
  std::vector<float> p(params, params + n);
  std::vector<uint16_t> w;
  pack_weights(p, w);
  float b[16 + 16 + 1];
  std::copy(p.begin() + OFF_B1, p.begin() + OFF_B1 + 16, b);
  std::copy(p.begin() + OFF_B2, p.begin() + OFF_B2 + 16, b + 16);
  b[32] = p[OFF_B3];
  if (L.wbf.ensure(w.size() * 2) != hipSuccess || L.bias.ensure(sizeof(b)) != hipSuccess ||
      L.master.ensure(size_t(n) * 4) != hipSuccess)
    return ctx->fail(RSG_ERR_HIP, "lpc: allocation failed");
  RSG_HIP(hipMemcpyAsync(L.wbf.p, w.data(), w.size() * 2, hipMemcpyHostToDevice, ctx->stream));
  RSG_HIP(hipMemcpyAsync(L.bias.p, b, sizeof(b), hipMemcpyHostToDevice, ctx->stream));
  RSG_HIP(hipMemcpyAsync(L.master.p, p.data(), size_t(n) * 4, hipMemcpyHostToDevice, ctx->stream));
  RSG_HIP(hipStreamSynchronize(ctx->stream));
  L.have_params = true;
  return RSG_OK;
}

int lpc_get_params(rsg_ctx *ctx, float *params) {
  LpcState &L = ctx->lpc;
  if (!L.have_params) return ctx->fail(RSG_ERR_STATE, "lpc: no parameters");
  RSG_HIP(hipMemcpyAsync(params, L.master.p, size_t(lpc_param_count()) * 4, hipMemcpyDeviceToHost, ctx->stream));
  RSG_HIP(hipStreamSynchronize(ctx->stream));
  return RSG_OK;
}

// v = (Vloc - mean) / std of the context's current Vloc, FP32
int lpc_set_potential(rsg_ctx *ctx, const double *vloc_host) {
  LpcState &L = ctx->lpc;
  const int64_t N = ctx->N;
  std::vector<double> v(vloc_host, vloc_host + N);
  double m = 0.0, q = 0.0;
  for (double x : v) m += x;
  m /= double(N);
  for (double x : v) q += (x - m) * (x - m);
  const double sd = std::sqrt(q / double(N)) + 1e-30;
  std::vector<float> f(static_cast<size_t>(N));
  for (int64_t i = 0; i < N; ++i) f[size_t(i)] = float((v[size_t(i)] - m) / sd);
  if (L.vnorm.ensure(size_t(N) * 4) != hipSuccess) return ctx->fail(RSG_ERR_HIP, "lpc: allocation failed");
  RSG_HIP(hipMemcpyAsync(L.vnorm.p, f.data(), size_t(N) * 4, hipMemcpyHostToDevice, ctx->stream));
  RSG_HIP(hipStreamSynchronize(ctx->stream));
  L.have_v = true;
  L.vN = N;
  return RSG_OK;
}

namespace {

int ensure_acts(rsg_ctx *ctx, int nsamp, bool training) {
  LpcState &L = ctx->lpc;
  const size_t N = size_t(ctx->N), ns = size_t(nsamp);
  bool ok = L.x0.ensure(ns * N * 4) == hipSuccess && L.a1.ensure(ns * N * 32) == hipSuccess &&
            L.a2.ensure(ns * N * 32) == hipSuccess && L.sval.ensure(ns * 4 + 256) == hipSuccess &&
            L.gg.ensure(ns * 8 + 256) == hipSuccess && L.y.ensure(ns * N * 4) == hipSuccess;
  if (training)
    ok = ok && L.dyb.ensure(ns * N * 2) == hipSuccess && L.dz1.ensure(ns * N * 32) == hipSuccess &&
         L.dz2.ensure(ns * N * 32) == hipSuccess;
  return ok ? RSG_OK : ctx->fail(RSG_ERR_HIP, "lpc: activation allocation failed");
}

template <int CIN, int KP, int MODE, typename T>
void launch_conv(rsg_ctx *ctx, int nsamp, const uint16_t *in, int64_t in_stride, const uint16_t *w,
                 const float *bias, uint16_t *out, const uint16_t *mask, float *yout, T *pg, int64_t ldg,
                 const float *sval) {
  const Grid3 g{ctx->n[0], ctx->n[1], ctx->n[2]};
  const int ntg = (g.n1 * g.n2 + 16 * kWaves - 1) / (16 * kWaves);
  // whole z-columns where they fill the chip (4 waves a SIMD: 1024 blocks),
  // else runs of at least four planes (each run reads two planes more)
  const int64_t cols = int64_t(ntg) * nsamp;
  int nzr = int(std::min<int64_t>(std::max(1, g.n3 / 4), (2048 + cols - 1) / cols));
  const int zlen = (g.n3 + nzr - 1) / nzr;
  nzr = (g.n3 + zlen - 1) / zlen;
  hipLaunchKernelGGL((k_conv<CIN, KP, MODE, T>), dim3(unsigned(cols * nzr)), dim3(64 * kWaves), 0, ctx->stream, g,
                     ctx->N, zlen, nzr, ntg, in, in_stride, w, bias, out, mask, yout, pg, ldg, sval);
}

// forward through all layers for nsamp samples g[smp*ldg + p]; y -> L.y;
// pg (if non-null) <- g + s y
template <typename T>
int forward_t(rsg_ctx *ctx, const T *g, int64_t ldg, int nsamp, T *pg, bool training) {
  LpcState &L = ctx->lpc;
  if (!L.have_params || !L.have_v || L.vN != ctx->N)
    return ctx->fail(RSG_ERR_STATE, "lpc: parameters or potential not set for this grid");
  int rc = ensure_acts(ctx, nsamp, training);
  if (rc) return rc;
  const int64_t N = ctx->N;
  // s = rms(g); multidot takes blocks with leading dimension N, so a
  // padded ldg goes one sample per call
  {
    if (ldg == N) {
      const T *xp[1] = {g}, *yp[1] = {g};
      if ((rc = multidot(ctx, 1, xp, yp, nsamp, 1.0, L.gg.as<double>()))) return rc;
    } else {
      for (int s = 0; s < nsamp; ++s) {
        const T *xp[1] = {g + int64_t(s) * ldg}, *yp[1] = {g + int64_t(s) * ldg};
        if ((rc = multidot(ctx, 1, xp, yp, 1, 1.0, L.gg.as<double>() + s))) return rc;
      }
    }
  }
  hipLaunchKernelGGL(k_rms, dim3((nsamp + 63) / 64), dim3(64), 0, ctx->stream, L.gg.as<double>(), nsamp, N,
                     L.sval.as<float>());
  hipLaunchKernelGGL((k_prep<T>), dim3(unsigned((N + 255) / 256), nsamp), dim3(256), 0, ctx->stream, g, ldg,
                     L.vnorm.as<float>(), L.sval.as<float>(), N, L.x0.as<uint16_t>());
  const uint16_t *w1 = L.wbf.as<uint16_t>(), *w2 = w1 + 16 * KP1, *w3 = w2 + 16 * KP2;
  const float *b = L.bias.as<float>();
  launch_conv<2, KP1, kReluOut, T>(ctx, nsamp, L.x0.as<uint16_t>(), N * 2, w1, b, L.a1.as<uint16_t>(), nullptr,
                                   nullptr, nullptr, 0, nullptr);
  launch_conv<16, KP2, kReluOut, T>(ctx, nsamp, L.a1.as<uint16_t>(), N * 16, w2, b + 16, L.a2.as<uint16_t>(),
                                    nullptr, nullptr, nullptr, 0, nullptr);
  launch_conv<16, KP3, kFinalOut, T>(ctx, nsamp, L.a2.as<uint16_t>(), N * 16, w3, b + 32, nullptr, nullptr,
                                     L.y.as<float>(), pg, ldg, L.sval.as<float>());
  RSG_HIP(hipGetLastError());
  return RSG_OK;
}

// quads of a line: one in front, the 16-point chunks, one behind
int quads_per_line(const rsg_ctx *ctx) { return 4 * ((ctx->n[0] + 15) / 16) + 2; }

// Samples whose quad layouts are held at once: both buffers, at the 16
// channels that each holds at some layer, within 1 GiB; at least one sample.
// The layout takes 1.6 times the field for 36 points a line, 2.4 times for
// 17; a batch of 16 samples of 36^3 points takes 74 MB.
constexpr int64_t kQuadBytes = int64_t(1) << 30;
int quad_samples(const rsg_ctx *ctx, int nsamp) {
  const int64_t per = int64_t(ctx->n[1]) * ctx->n[2] * quads_per_line(ctx) * 2 * 16 * 8;
  return int(std::max<int64_t>(1, std::min<int64_t>(nsamp, kQuadBytes / per)));
}

template <int C> void to_quads(rsg_ctx *ctx, int nsamp, const uint16_t *in, int wrap, uint16_t *out) {
  const int64_t nrow = int64_t(ctx->n[1]) * ctx->n[2] * nsamp;
  const int nq = quads_per_line(ctx);
  // a launch holds fewer than 2^32 threads in a dimension
  const int64_t nblk = (nrow * nq * C + 255) / 256, gx = std::min<int64_t>(nblk, int64_t(1) << 23);
  hipLaunchKernelGGL((k_quads<C>), dim3(unsigned(gx), unsigned((nblk + gx - 1) / gx)), dim3(256), 0, ctx->stream, in,
                     nrow, ctx->n[0], nq, wrap, out);
}

// gradient of a layer's weights into out and of its biases into db; the
// samples go through the quad buffers in groups, whose partial sums lie one
// after another
template <int CIN, int KP, int COUT>
int weight_grad(rsg_ctx *ctx, int nsamp, const uint16_t *in, const uint16_t *dz, float *out, float *db) {
  LpcState &L = ctx->lpc;
  const Grid3 g{ctx->n[0], ctx->n[1], ctx->n[2]};
  const int64_t N = ctx->N, n23 = int64_t(g.n2) * g.n3, total = N * nsamp;
  const int nq = quads_per_line(ctx), per = quad_samples(ctx, nsamp);
  auto blocks = [&](int ns) { return int(std::min<int64_t>(512, (n23 * ns + 15) / 16)); };
  const int64_t nblk = int64_t(nsamp / per) * blocks(per) + (nsamp % per ? blocks(nsamp % per) : 0);
  const unsigned nbb = unsigned(std::min<int64_t>(512, (total * COUT + 8 * 256 - 1) / (8 * 256)));
  if (L.part.ensure(std::max(size_t(nblk) * 16 * KP, size_t(nbb) * COUT) * 4) != hipSuccess ||
      L.xq.ensure(size_t(n23) * per * nq * CIN * 8) != hipSuccess ||
      L.dq.ensure(size_t(n23) * per * nq * COUT * 8) != hipSuccess)
    return ctx->fail(RSG_ERR_HIP, "lpc: allocation failed");
  float *part = L.part.as<float>();
  int64_t b0 = 0;
  for (int s0 = 0; s0 < nsamp; s0 += per) {
    const int ns = std::min(per, nsamp - s0), nb = blocks(ns);
    to_quads<CIN>(ctx, ns, in + int64_t(s0) * N * CIN, 1, L.xq.as<uint16_t>());
    to_quads<COUT>(ctx, ns, dz + int64_t(s0) * N * COUT, 0, L.dq.as<uint16_t>());
    hipLaunchKernelGGL((k_conv_dw<CIN, KP, COUT>), dim3(nb), dim3(256), 0, ctx->stream, g, ns, L.xq.as<uint16_t>(),
                       L.dq.as<uint16_t>(), nq, part + b0 * 16 * KP);
    b0 += nb;
  }
  const int len = 16 * KP;
  hipLaunchKernelGGL(k_sum_parts, dim3((len + 63) / 64), dim3(1024), 0, ctx->stream, part, int(nblk), len, out);
  hipLaunchKernelGGL(k_bias_grad<COUT>, dim3(nbb), dim3(256), 0, ctx->stream, dz, total, part);
  hipLaunchKernelGGL(k_sum_parts, dim3(1), dim3(1024), 0, ctx->stream, part, int(nbb), COUT, db);
  return RSG_OK;
}

}  // namespace

// bands per forward pass: activations take 68 bytes per point and band
static int apply_chunk(const rsg_ctx *ctx, int nb) {
  const size_t per = size_t(ctx->N) * 72;
  return int(std::max<size_t>(1, std::min<size_t>(size_t(nb), (size_t(4) << 30) / per)));
}

int lpc_apply(rsg_ctx *ctx, const void *g, void *pg, int64_t ld, int nb, int precision) {
  if (precision != 64 && precision != 32) return ctx->fail(RSG_ERR_ARG, "lpc: precision must be 64 or 32");
  if (ld < ctx->N || nb < 0) return ctx->fail(RSG_ERR_ARG, "lpc: bad ld or nb");
  const int ch = apply_chunk(ctx, std::max(nb, 1));
  for (int b0 = 0; b0 < nb; b0 += ch) {
    const int n = std::min(ch, nb - b0);
    int rc;
    if (precision == 64)
      rc = forward_t<double>(ctx, static_cast<const double *>(g) + int64_t(b0) * ld, ld, n,
                             static_cast<double *>(pg) + int64_t(b0) * ld, false);
    else
      rc = forward_t<float>(ctx, static_cast<const float *>(g) + int64_t(b0) * ld, ld, n,
                            static_cast<float *>(pg) + int64_t(b0) * ld, false);
    if (rc) return rc;
  }
  return RSG_OK;
}

// One training step on nsamp samples (FP32 residuals g and targets t, each
// N x nsamp column-major): forward, loss against kappa t, backward,
// optional Adam update.  grads (host, may be NULL) receives the gradient in
// the parameter layout.
int lpc_train_step(rsg_ctx *ctx, const float *g, const float *t, int nsamp, float kappa, float lr, double *loss,
                   float *grads) {
  LpcState &L = ctx->lpc;
  int rc = forward_t<float>(ctx, g, ctx->N, nsamp, nullptr, true);
  if (rc) return rc;
  const int64_t N = ctx->N;
  const int np = lpc_param_count();
  if (L.lsum.ensure(64) != hipSuccess || L.grad.ensure(size_t(16) * (KP1 + KP2 + KP3) * 4 + 256) != hipSuccess)
    return ctx->fail(RSG_ERR_HIP, "lpc: allocation failed");
  RSG_HIP(hipMemsetAsync(L.lsum.p, 0, 64, ctx->stream));
  const double inv = 1.0 / (double(N) * nsamp);
  hipLaunchKernelGGL(k_loss, dim3(unsigned((N + 255) / 256), nsamp), dim3(256), 0, ctx->stream, t, L.y.as<float>(),
                     L.sval.as<float>(), kappa, N, inv, L.dyb.as<uint16_t>(), L.lsum.as<double>());
  const uint16_t *w1 = L.wbf.as<uint16_t>(), *w2 = w1 + 16 * KP1, *w3 = w2 + 16 * KP2, *w2t = w3 + 16 * KP3,
                 *w3t = w2t + 16 * KP2;
  // dz2 = (W3' * dy) masked by a2 > 0 ; dz1 = (W2' * dz2) masked by a1 > 0
  launch_conv<1, KP3T, kMaskedGrad, float>(ctx, nsamp, L.dyb.as<uint16_t>(), N, w3t, nullptr, L.dz2.as<uint16_t>(),
                                           L.a2.as<uint16_t>(), nullptr, nullptr, 0, nullptr);
  launch_conv<16, KP2, kMaskedGrad, float>(ctx, nsamp, L.dz2.as<uint16_t>(), N * 16, w2t, nullptr,
                                           L.dz1.as<uint16_t>(), L.a1.as<uint16_t>(), nullptr, nullptr, 0, nullptr);
  // weight gradients into grad = [G1 16 x KP1 | G2 16 x KP2 | G3 16 x KP3 (row 0)]
  float *G = L.grad.as<float>(), *db = G + 16 * (KP1 + KP2 + KP3);
  if ((rc = weight_grad<2, KP1, 16>(ctx, nsamp, L.x0.as<uint16_t>(), L.dz1.as<uint16_t>(), G, db))) return rc;
  if ((rc = weight_grad<16, KP2, 16>(ctx, nsamp, L.a1.as<uint16_t>(), L.dz2.as<uint16_t>(), G + 16 * KP1, db + 16)))
    return rc;
  if ((rc = weight_grad<16, KP3, 1>(ctx, nsamp, L.a2.as<uint16_t>(), L.dyb.as<uint16_t>(), G + 16 * (KP1 + KP2),
                                    db + 32)))
    return rc;
  RSG_HIP(hipGetLastError());
  // gather into the parameter layout on the host (8241 floats)
  std::vector<float> Gh(size_t(16) * (KP1 + KP2 + KP3) + 33);
  RSG_HIP(hipMemcpyAsync(Gh.data(), G, Gh.size() * 4, hipMemcpyDeviceToHost, ctx->stream));
  double lh = 0.0;
  RSG_HIP(hipMemcpyAsync(&lh, L.lsum.p, 8, hipMemcpyDeviceToHost, ctx->stream));
  RSG_HIP(hipStreamSynchronize(ctx->stream));
  if (loss) *loss = lh;
  std::vector<float> gp(size_t(np), 0.f);
  const float *g1 = Gh.data(), *g2 = g1 + 16 * KP1, *g3 = g2 + 16 * KP2, *gb = g3 + 16 * KP3;
  for (int co = 0; co < 16; ++co)
    for (int ci = 0; ci < 2; ++ci)
      for (int tp = 0; tp < 27; ++tp) gp[size_t(OFF_W1 + (co * 2 + ci) * 27 + tp)] = g1[co * KP1 + tp * 2 + ci];
  for (int co = 0; co < 16; ++co)
    for (int ci = 0; ci < 16; ++ci)
      for (int tp = 0; tp < 27; ++tp) gp[size_t(OFF_W2 + (co * 16 + ci) * 27 + tp)] = g2[co * KP2 + tp * 16 + ci];
  for (int ci = 0; ci < 16; ++ci)
    for (int tp = 0; tp < 27; ++tp) gp[size_t(OFF_W3 + ci * 27 + tp)] = g3[0 * KP3 + tp * 16 + ci];
  for (int c = 0; c < 16; ++c) gp[size_t(OFF_B1 + c)] = gb[c];
  for (int c = 0; c < 16; ++c) gp[size_t(OFF_B2 + c)] = gb[16 + c];
  gp[size_t(OFF_B3)] = gb[32];
  if (grads) std::copy(gp.begin(), gp.end(), grads);
  if (lr > 0.f) {
    if (L.mom1.ensure(size_t(np) * 4) != hipSuccess || L.mom2.ensure(size_t(np) * 4) != hipSuccess)
      return ctx->fail(RSG_ERR_HIP, "lpc: allocation failed");
    if (L.adam_t == 0) {
      RSG_HIP(hipMemsetAsync(L.mom1.p, 0, size_t(np) * 4, ctx->stream));
      RSG_HIP(hipMemsetAsync(L.mom2.p, 0, size_t(np) * 4, ctx->stream));
    }
    ++L.adam_t;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - std::pow(b1, float(L.adam_t)), c2 = 1.f - std::pow(b2, float(L.adam_t));
    // the gradient in parameter layout goes up once; the update runs on the device
    RSG_HIP(hipMemcpyAsync(G, gp.data(), size_t(np) * 4, hipMemcpyHostToDevice, ctx->stream));
    hipLaunchKernelGGL(k_adam, dim3((np + 255) / 256), dim3(256), 0, ctx->stream, L.master.as<float>(), G,
                       L.mom1.as<float>(), L.mom2.as<float>(), np, lr, b1, b2, 1e-8f, c1, c2);
    std::vector<float> p(static_cast<size_t>(np));
    RSG_HIP(hipMemcpyAsync(p.data(), L.master.p, size_t(np) * 4, hipMemcpyDeviceToHost, ctx->stream));
    RSG_HIP(hipStreamSynchronize(ctx->stream));
    return lpc_set_params(ctx, p.data());
  }
  return RSG_OK;
}

int lpc_reset_optimizer(rsg_ctx *ctx) {
  ctx->lpc.adam_t = 0;
  return RSG_OK;
}

}  // namespace rsg
