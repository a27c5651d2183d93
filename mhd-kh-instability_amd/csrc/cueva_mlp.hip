// Learned primitive recovery: training and inference kernels of the
// 3 -> 32 -> 32 -> 2 start-point MLP (cueva_mlp.hpp) and the primitive
// recovery that uses it.
//
//  - k_mlp_grad: forward (BF16) and backward (FP32) on the matrix cores; the
//    gradient of the mean squared error over a sample range, w.r.t. the FP32
//    master weights (the forward uses their BF16 rounding), as partial sums.
//  - k_mlp_adam: their sum, and one Adam update of the master weights.
//  - k_mlp_forward: normalised outputs for normalised inputs (tests).
//  - k_c2p_learned: per cell, the network's start for W, at most two FP64 Newton
//    steps on the quartic of 12_varprimitive.f95:245-296, acceptance when the
//    relative quartic residual is <= 1e-10, W >= 1 and the state it implies is
//    physical and agrees with the network's pressure, otherwise the Cardano
//    path of the reference; then the reference's pressure loop, fix-ups and
//    velocities (12_varprimitive.f95:510-696).  Cardano fallbacks are counted.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include "cueva.h"
#include "cueva_common.hpp"
#include "cueva_mlp.hpp"
#include "cueva_update.hpp"

namespace cueva {
namespace mlp {

constexpr int GRAD_WAVES = 4;                    // wavefronts of a k_mlp_grad block, one 16-sample tile each at a time
constexpr int GRAD_TILE = 16 * GRAD_WAVES;       // samples a block takes per pass
constexpr int GRAD_BLOCKS = 256;                 // blocks (partial gradients) at most
constexpr int GRAD_PITCH = (NPARAM + 63) / 64 * 64;  // floats of one partial gradient
constexpr int TP = 17;                           // padded LDS row of 16 samples

__device__ inline f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Partial gradients of sum over [off, off+n) of |y - t|^2 / n_total: block b's
// sum to part[b], its share of the loss to lossp[b].
//
// All matrix products run on the matrix cores: the forward in BF16 as the
// inference does, the backward in FP32 (v_mfma_f32_16x16x4_f32), as the
// gradient was computed before.  A wavefront holds a tile of 16 samples: lane
// (r, kb) has units 16m + 4kb + i of sample r, which is the B operand of
// dz1 = W2^T dz2 as it stands (the four k of one product are the units
// 16m + 4kb + i of one (m, i)); the weight gradients contract over the
// samples and take dz2, dz1, h1, h2 back from LDS transposed.  One sample per
// thread with the contractions as LDS loops took 85 us for a batch of 4096,
// bound by the LDS latency of two wavefronts on 32 CUs; now 64 blocks of four
// tiles, 7 us, and the update 4.9 -> 4 us (16.4 us a step of 4096 samples with its
// launches, was 93.6).
__global__ void __launch_bounds__(64 * GRAD_WAVES) k_mlp_grad(const float* __restrict__ p, const float* __restrict__ X,
                                                              const float* __restrict__ Y, int64_t off, int64_t n,
                                                              float inv_total, float* __restrict__ part,
                                                              double* __restrict__ lossp) {
  struct Wave {
    float dz2[NH][TP], dz1[NH][TP], h1[NH][TP], h2[NH][TP];
    float x[4][TP];   // x0 x1 x2 and 1 (the bias column)
    float dy[2][TP];
  };
  __shared__ union {
    Wave w[GRAD_WAVES];
    float g[GRAD_WAVES][GRAD_PITCH];  // after the tiles: each wavefront's gradient
  } sh;
  __shared__ double lsum[GRAD_WAVES];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, r = lane & 15, kb = lane >> 4;
  Wave& w = sh.w[wv];
  const Operands o = load_operands(p, lane);
  float w2t[2][4][2], w3[2][2][4];  // W2[16m+4kb+i][16mo+r], W3[o][16m+4kb+i], as the forward rounds them
#pragma unroll
  for (int m = 0; m < 2; m++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
      for (int mo = 0; mo < 2; mo++) w2t[m][i][mo] = bf16_round(p[OFF_W2 + (16 * m + 4 * kb + i) * NH + 16 * mo + r]);
#pragma unroll
      for (int q = 0; q < NOUT; q++) w3[q][m][i] = bf16_round(p[OFF_W3 + q * NH + 16 * m + 4 * kb + i]);
    }
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 g2[2][2] = {{zero, zero}, {zero, zero}}, g1[2] = {zero, zero}, gb2[2] = {zero, zero}, g3[2] = {zero, zero};
  float gb3[2] = {0.0f, 0.0f};
  double l2 = 0.0;
  const int64_t step = (int64_t)gridDim.x * GRAD_TILE;
  for (int64_t t0 = (int64_t)blockIdx.x * GRAD_TILE; t0 < n; t0 += step) {  // uniform over the block
    const int64_t c = t0 + 16 * wv + r;  // this lane's sample
    const bool valid = c < n;
    float x0 = 0.0f, x1 = 0.0f, x2 = 0.0f, y0 = 0.0f, y1 = 0.0f;
    if (valid) {
      x0 = X[(off + c) * 3 + 0]; x1 = X[(off + c) * 3 + 1]; x2 = X[(off + c) * 3 + 2];
      y0 = Y[(off + c) * 2 + 0]; y1 = Y[(off + c) * 2 + 1];
    }
    const TileAct a = forward_tile(o, lane, 0, x0, x1, x2);  // tile 0: every lane passes its own sample r
    const float e0 = __shfl(a.y[0], r, 64) - y0, e1 = __shfl(a.y[1], r, 64) - y1;
    const float dy0 = valid ? 2.0f * e0 * inv_total : 0.0f, dy1 = valid ? 2.0f * e1 * inv_total : 0.0f;
    if (valid && kb == 0) {
      l2 += ((double)e0 * e0 + (double)e1 * e1) * inv_total;
      gb3[0] += dy0;
      gb3[1] += dy1;
    }
    float dz2[2][4];
    f32x4 d1[2] = {zero, zero};
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        dz2[m][i] = (dy0 * w3[0][m][i] + dy1 * w3[1][m][i]) * (1.0f - a.h2[m][i] * a.h2[m][i]);
#pragma unroll
        for (int mo = 0; mo < 2; mo++) d1[mo] = mfma4(w2t[m][i][mo], dz2[m][i], d1[mo]);
      }
    __syncthreads();  // the previous pass has read its rows
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int u = 16 * m + 4 * kb + i;
        w.dz2[u][r] = dz2[m][i];
        w.dz1[u][r] = d1[m][i] * (1.0f - a.h1[m][i] * a.h1[m][i]);
        w.h1[u][r] = bf16_round(a.h1[m][i]);
        w.h2[u][r] = bf16_round(a.h2[m][i]);
      }
    if (kb == 0) {
      w.x[0][r] = bf16_round(x0); w.x[1][r] = bf16_round(x1); w.x[2][r] = bf16_round(x2);
      w.x[3][r] = 1.0f;
      w.dy[0][r] = dy0; w.dy[1][r] = dy1;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; q++) {  // samples 4q .. 4q+3
      const int s = 4 * q + kb;
      const float bx = r < 4 ? w.x[r & 3][s] : 0.0f, by = r < 2 ? w.dy[r & 1][s] : 0.0f, one = r == 0 ? 1.0f : 0.0f;
      const float bh[2] = {w.h1[r][s], w.h1[16 + r][s]};
#pragma unroll
      for (int mo = 0; mo < 2; mo++) {
        const float a2 = w.dz2[16 * mo + r][s];
#pragma unroll
        for (int mi = 0; mi < 2; mi++) g2[mo][mi] = mfma4(a2, bh[mi], g2[mo][mi]);
        gb2[mo] = mfma4(a2, one, gb2[mo]);
        g1[mo] = mfma4(w.dz1[16 * mo + r][s], bx, g1[mo]);
        g3[mo] = mfma4(w.h2[16 * mo + r][s], by, g3[mo]);
      }
    }
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    l2 += __shfl_down(l2, d, 64);
    if (d < 16) {  // the samples sit in lanes 0..15
      gb3[0] += __shfl_down(gb3[0], d, 64);
      gb3[1] += __shfl_down(gb3[1], d, 64);
    }
  }
  __syncthreads();  // the tile rows give way to the wavefronts' gradients
  float* g = sh.g[wv];
#pragma unroll
  for (int mo = 0; mo < 2; mo++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int h = 16 * mo + 4 * kb + i;
#pragma unroll
      for (int mi = 0; mi < 2; mi++) g[OFF_W2 + h * NH + 16 * mi + r] = g2[mo][mi][i];
      if (r < NIN) g[OFF_W1 + h * NIN + r] = g1[mo][i];
      if (r == NIN) g[OFF_B1 + h] = g1[mo][i];
      if (r == 0) g[OFF_B2 + h] = gb2[mo][i];
      if (r < NOUT) g[OFF_W3 + r * NH + h] = g3[mo][i];
    }
  if (lane == 0) {
    g[OFF_B3 + 0] = gb3[0];
    g[OFF_B3 + 1] = gb3[1];
    lsum[wv] = l2;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < NPARAM; e += 64 * GRAD_WAVES) {
    float v = sh.g[0][e];
#pragma unroll
    for (int k = 1; k < GRAD_WAVES; k++) v += sh.g[k][e];
    part[(int64_t)blockIdx.x * GRAD_PITCH + e] = v;
  }
  if (threadIdx.x == 0) {
    double v = lsum[0];
    for (int k = 1; k < GRAD_WAVES; k++) v += lsum[k];
    lossp[blockIdx.x] = v;
  }
}

// The gradient from the blocks' partial sums, in a fixed order (the same every
// run), and with ADAM one update of the master weights.  64 parameters per
// block, four threads to a parameter, so that the partial sums are read by 20
// blocks; add: *loss += the batch's loss, else =.
template <bool ADAM>
__global__ void __launch_bounds__(256) k_mlp_adam(float* __restrict__ p, const float* __restrict__ part,
                                                  const double* __restrict__ lossp, int nb, float* __restrict__ grad,
                                                  float* __restrict__ m1, float* __restrict__ m2,
                                                  double* __restrict__ loss, int add, float lr, float b1t, float b2t) {
  __shared__ float s[4][64];
  const int l = threadIdx.x & 63, q = threadIdx.x >> 6, e = (int)blockIdx.x * 64 + l;
  float g = 0.0f;
#pragma unroll 8
  for (int b = q; b < nb; b += 4) g += part[(int64_t)b * GRAD_PITCH + e];  // rows are padded to whole blocks
  s[q][l] = g;
  if (blockIdx.x == 0 && q == 1) {
    double v = 0.0;
    for (int b = l; b < nb; b += 64) v += lossp[b];
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_down(v, d, 64);
    if (l == 0) *loss = add ? *loss + v : v;
  }
  __syncthreads();
  if (q != 0 || e >= NPARAM) return;
  g = (s[0][l] + s[1][l]) + (s[2][l] + s[3][l]);
  if (!ADAM) {
    grad[e] = g;
    return;
  }
  const float b1 = 0.9f, b2 = 0.999f, eps = 1.0e-8f;
  float a = b1 * m1[e] + (1.0f - b1) * g;
  float v = b2 * m2[e] + (1.0f - b2) * g * g;
  m1[e] = a;
  m2[e] = v;
  float ah = a / (1.0f - b1t), vh = v / (1.0f - b2t);
  p[e] -= lr * ah / (sqrtf(vh) + eps);
}

__global__ void __launch_bounds__(256) k_mlp_forward(const float* __restrict__ p, const float* __restrict__ X,
                                                     int64_t n, float* __restrict__ Yo) {
  const int lane = threadIdx.x & 63;
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = c < n;
  float x0 = valid ? X[c * 3 + 0] : 0.0f, x1 = valid ? X[c * 3 + 1] : 0.0f, x2 = valid ? X[c * 3 + 2] : 0.0f;
  Operands o = load_operands(p, lane);
  float y0 = 0.0f, y1 = 0.0f;
  forward_wave(o, lane, x0, x1, x2, y0, y1);
  if (valid) {
    Yo[c * 2 + 0] = y0;
    Yo[c * 2 + 1] = y1;
  }
}

}  // namespace mlp

// ---------------------------------------------------------------------------
// learned primitive recovery over the interior, one thread per cell
// (STAGE0: also the next step's stage-0 state, as k_c2p<true>)
// ---------------------------------------------------------------------------
template <bool STAGE0>
__global__ void __launch_bounds__(256) k_c2p_learned(Geom g, Planes P, Scheme S, const float* __restrict__ wp,
                                                     StatusRef sr) {
  using namespace mlp;
  if (halted(sr)) return;
  const int lane = threadIdx.x & 63;
  const int i0 = (int)(blockIdx.x * 64 + threadIdx.x), j0 = (int)(blockIdx.y * 4 + threadIdx.y);
  const bool valid = i0 <= g.imax && j0 <= g.jmax;
  // the network runs wavefront-wide: points past the edge compute on an edge point
  const int i = i0 <= g.imax ? i0 : g.imax, j = j0 <= g.jmax ? j0 : g.jmax;
  const int64_t k = g.at(i, j);
  C2PIn in;
  in.d = P.c[C_D][k]; in.tau = P.c[C_TAU][k];
  in.sx = P.c[C_SX][k]; in.sy = P.c[C_SY][k]; in.sz = P.c[C_SZ][k];
  in.ex = P.p[P_EX][k]; in.ey = P.p[P_EY][k]; in.ez = P.p[P_EZ][k];
  in.bx = P.p[P_BX][k]; in.by = P.p[P_BY][k]; in.bz = P.p[P_BZ][k];
  in.vx0 = P.p[P_VX][k]; in.vy0 = P.p[P_VY][k]; in.vz0 = P.p[P_VZ][k];
  in.rho_old = P.p[P_RHO][k]; in.p_old = P.p[P_P][k];
  Operands o = load_operands(wp, lane);
  C2POut out;
  bool fallback = false;
  const int code = c2p_learned_cell(S.gamma, S.eps1, in, wp, o, lane, S.crmath != 0, out, fallback);
  if (!valid) return;
  if (fallback) atomicAdd(&sr.st->fallback, 1ULL);
  if (code) { report(sr, code, i, j, 1); return; }
  c2p_count(sr, i, j, out);
  c2p_store_out(P, S, k, out);
  if (STAGE0) stage0_after_c2p(P, S, k, in, out);
}

hipError_t launch_c2p_learned(hipStream_t s, const Geom& g, const Planes& P, const Scheme& S, const float* wp,
                              const StatusRef& sr, bool stage0) {
  // rows of 64 points, each starting at a multiple of 64 columns: whole cache lines
  const dim3 grid((unsigned)((g.imax + 64) / 64), (unsigned)((g.jmax + 4) / 4)), blk(64, 4);
  if (stage0)
    hipLaunchKernelGGL(k_c2p_learned<true>, grid, blk, 0, s, g, P, S, wp, sr);
  else
    hipLaunchKernelGGL(k_c2p_learned<false>, grid, blk, 0, s, g, P, S, wp, sr);
  return hipGetLastError();
}

}  // namespace cueva

// ---------------------------------------------------------------------------
// C ABI of the model (declared in include/cueva.h)
// ---------------------------------------------------------------------------
using namespace cueva;

struct cueva_mlp {
  float* p;      // packed parameters (NPACK)
  float* grad;   // NPARAM
  float* m1;     // Adam moments
  float* m2;
  double* loss;
  double* lossp;  // per block of k_mlp_grad: its share of the loss
  float* part;    // and its gradient (GRAD_PITCH floats)
  float* X;      // training inputs (3 per sample), normalised
  float* Y;      // training targets (2 per sample), normalised
  int64_t n, cap;
  int64_t t;     // Adam step count
  hipStream_t stream;
};

#define MCHK(x)                                   \
  do {                                            \
    if ((x) != hipSuccess) return CUEVA_E_HIP;    \
  } while (0)

extern "C" int cueva_mlp_create(cueva_mlp** out) {
  if (!out) return CUEVA_E_ARG;
  cueva_mlp* m = new cueva_mlp();
  const size_t head = sizeof(float) * (mlp::NPACK + 3 * mlp::NPARAM);
  const size_t bytes = head + sizeof(double) * (1 + mlp::GRAD_BLOCKS) +
                       sizeof(float) * (size_t)mlp::GRAD_BLOCKS * mlp::GRAD_PITCH;
  char* base;
  if (hipMalloc(&base, bytes) != hipSuccess) { delete m; return CUEVA_E_NOMEM; }
  m->p = (float*)base;
  m->grad = m->p + mlp::NPACK;
  m->m1 = m->grad + mlp::NPARAM;
  m->m2 = m->m1 + mlp::NPARAM;
  m->lossp = (double*)(base + head) + 1;
  m->part = (float*)(m->lossp + mlp::GRAD_BLOCKS);
  m->loss = (double*)(base + head);  // NPACK + 3 NPARAM floats = 20040 bytes: 8-byte aligned
  static_assert(((mlp::NPACK + 3 * mlp::NPARAM) * sizeof(float)) % 8 == 0, "loss alignment");
  if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess) {
    hipFree(base);
    delete m;
    return CUEVA_E_HIP;
  }
  if (hipMemsetAsync(base, 0, bytes, m->stream) != hipSuccess || hipStreamSynchronize(m->stream) != hipSuccess) {
    hipStreamDestroy(m->stream);
    hipFree(base);
    delete m;
    return CUEVA_E_HIP;
  }
  *out = m;
  return CUEVA_OK;
}

extern "C" int cueva_mlp_destroy(cueva_mlp* m) {
  if (!m) return CUEVA_E_ARG;
  hipStreamSynchronize(m->stream);
  hipFree(m->p);
  if (m->X) hipFree(m->X);
  hipStreamDestroy(m->stream);
  delete m;
  return CUEVA_OK;
}

extern "C" int cueva_mlp_set_params(cueva_mlp* m, const float* packed) {
  if (!m || !packed) return CUEVA_E_ARG;
  MCHK(hipMemcpyAsync(m->p, packed, sizeof(float) * mlp::NPACK, hipMemcpyHostToDevice, m->stream));
  MCHK(hipMemsetAsync(m->m1, 0, sizeof(float) * 2 * mlp::NPARAM, m->stream));
  MCHK(hipStreamSynchronize(m->stream));
  m->t = 0;
  return CUEVA_OK;
}

extern "C" int cueva_mlp_get_params(cueva_mlp* m, float* packed) {
  if (!m || !packed) return CUEVA_E_ARG;
  MCHK(hipMemcpyAsync(packed, m->p, sizeof(float) * mlp::NPACK, hipMemcpyDeviceToHost, m->stream));
  MCHK(hipStreamSynchronize(m->stream));
  return CUEVA_OK;
}

extern "C" int cueva_mlp_set_data(cueva_mlp* m, const float* x, const float* y, int64_t n) {
  if (!m || !x || !y || n <= 0) return CUEVA_E_ARG;
  if (n > m->cap) {
    if (m->X) hipFree(m->X);
    m->X = nullptr;
    if (hipMalloc(&m->X, sizeof(float) * 5 * (size_t)n) != hipSuccess) { m->cap = 0; return CUEVA_E_NOMEM; }
    m->cap = n;
  }
  m->Y = m->X + 3 * n;
  m->n = n;
  MCHK(hipMemcpyAsync(m->X, x, sizeof(float) * 3 * (size_t)n, hipMemcpyHostToDevice, m->stream));
  MCHK(hipMemcpyAsync(m->Y, y, sizeof(float) * 2 * (size_t)n, hipMemcpyHostToDevice, m->stream));
  MCHK(hipStreamSynchronize(m->stream));
  return CUEVA_OK;
}

// partial gradients of samples [off, off + cnt); returns their number
static int launch_grad(cueva_mlp* m, int64_t off, int64_t cnt) {
  const int64_t want = (cnt + mlp::GRAD_TILE - 1) / mlp::GRAD_TILE;
  const int nb = (int)(want < mlp::GRAD_BLOCKS ? want : mlp::GRAD_BLOCKS);
  hipLaunchKernelGGL(mlp::k_mlp_grad, dim3((unsigned)nb), dim3(64 * mlp::GRAD_WAVES), 0, m->stream, (const float*)m->p,
                     (const float*)m->X, (const float*)m->Y, off, cnt, 1.0f / (float)cnt, m->part, m->lossp);
  return nb;
}

extern "C" int cueva_mlp_grad(cueva_mlp* m, int64_t off, int64_t cnt, float* grad_out, double* loss_out) {
  if (!m || off < 0 || cnt <= 0 || off + cnt > m->n) return CUEVA_E_ARG;
  const int nb = launch_grad(m, off, cnt);
  hipLaunchKernelGGL(mlp::k_mlp_adam<false>, dim3(mlp::GRAD_PITCH / 64), dim3(256), 0, m->stream, m->p,
                     (const float*)m->part, (const double*)m->lossp, nb, m->grad, m->m1, m->m2, m->loss, 0, 0.0f, 0.0f,
                     0.0f);
  MCHK(hipGetLastError());
  if (grad_out) MCHK(hipMemcpyAsync(grad_out, m->grad, sizeof(float) * mlp::NPARAM, hipMemcpyDeviceToHost, m->stream));
  if (loss_out) MCHK(hipMemcpyAsync(loss_out, m->loss, sizeof(double), hipMemcpyDeviceToHost, m->stream));
  MCHK(hipStreamSynchronize(m->stream));
  return CUEVA_OK;
}

extern "C" int cueva_mlp_train(cueva_mlp* m, int64_t batch, int steps, float lr, double* loss_out) {
  if (!m || batch <= 0 || steps <= 0 || m->n < batch) return CUEVA_E_ARG;
  const int64_t nb = m->n / batch;
  for (int s = 0; s < steps; s++) {
    const int64_t off = ((m->t) % nb) * batch;
    const int parts = launch_grad(m, off, batch);
    m->t++;
    const float b1t = powf(0.9f, (float)m->t), b2t = powf(0.999f, (float)m->t);
    hipLaunchKernelGGL(mlp::k_mlp_adam<true>, dim3(mlp::GRAD_PITCH / 64), dim3(256), 0, m->stream, m->p,
                       (const float*)m->part, (const double*)m->lossp, parts, m->grad, m->m1, m->m2, m->loss, s > 0, lr,
                       b1t, b2t);
  }
  MCHK(hipGetLastError());
  double l = 0.0;
  MCHK(hipMemcpyAsync(&l, m->loss, sizeof(double), hipMemcpyDeviceToHost, m->stream));
  MCHK(hipStreamSynchronize(m->stream));
  if (loss_out) *loss_out = l / steps;
  return CUEVA_OK;
}

extern "C" int cueva_mlp_forward(cueva_mlp* m, const float* x, int64_t n, float* y) {
  if (!m || !x || !y || n <= 0) return CUEVA_E_ARG;
  float* buf;
  if (hipMalloc(&buf, sizeof(float) * 5 * (size_t)n) != hipSuccess) return CUEVA_E_NOMEM;
  int rc = CUEVA_OK;
  if (hipMemcpyAsync(buf, x, sizeof(float) * 3 * (size_t)n, hipMemcpyHostToDevice, m->stream) != hipSuccess)
    rc = CUEVA_E_HIP;
  if (!rc) {
    hipLaunchKernelGGL(mlp::k_mlp_forward, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, m->stream,
                       (const float*)m->p, (const float*)buf, n, buf + 3 * n);
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(y, buf + 3 * n, sizeof(float) * 2 * (size_t)n, hipMemcpyDeviceToHost, m->stream) != hipSuccess ||
        hipStreamSynchronize(m->stream) != hipSuccess)
      rc = CUEVA_E_HIP;
  }
  hipStreamSynchronize(m->stream);
  hipFree(buf);
  return rc;
}
