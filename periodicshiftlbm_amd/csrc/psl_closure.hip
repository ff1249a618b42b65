// Learned eddy-viscosity closure: training (FP32), data preparation from a
// fine-grid run, inference (bf16 matrix cores) and the C ABI.
//
// No reference counterpart (the reference's LES model is Smagorinsky,
// include/cellFunctions.h:157-198).  Pipeline:
//   1. a fine periodic grid (this solver) gives rho and u per cell
//      (psl_get_macroscopic);
//   2. k_les_filter: box filter of width r -> coarse rho, Favre velocity and
//      subgrid stress tau = <rho u u>/<rho> - u~ u~;
//   3. k_les_targets: coarse strain rate S by periodic central differences;
//      target nu_t* = max(0, -dev(tau):S / (2 S:S)); the non-equilibrium
//      second moments a perfect closure would produce on the coarse grid,
//      Pi = -(2/3) rho tau_eff S with tau_eff = 3 (nu + nu_t*) + 1/2, and from
//      them the raw closure inputs (closure_features);
//   4. training: mean-squared error of y against nu_t* / NU_SCALE, Adam,
//      mini-batches drawn by a counter-based generator; forward, backward and
//      gradient sums of 64 rows per workgroup in k_mlp_batch, their total and
//      the update in k_mlp_adam (fixed summation order);
//   5. inference inside the step (closure_wave, psl_closure.h).
#include "psl_closure.h"
#include "psl_stream.h"

#include <cmath>
#include <cstring>

namespace psl {

// ------------------------------------------------------------ training
// One iteration is two launches.  What bounds it is latency, not work (a
// 16384-row batch is 0.13 GFLOP): with one row per thread and its 32-wide
// layers in scratch the forward/backward pass took 42 us, the gradient pass
// another 16 us over activations written to memory, and the update 59 us in
// 256 serial additions per parameter, 125 us with the index launch.  Here a
// workgroup takes 64 rows through both passes and their gradients in LDS and
// the update adds the workgroups' sums 16 ways at once: 17 us per iteration.
constexpr int CHUNK = 64;     // rows per workgroup
constexpr int ROWS = 64 + 4;  // LDS row length: 16-byte aligned, rows 4 banks apart

// The rows of a mini-batch: row b of iteration `step` is splitmix64(seed, step,
// b) mod n, or b itself (draw = false).
struct BatchDraw {
  bool draw;
  uint32_t n;
  uint64_t recip;  // floor((2^64 - 1) / n)
  uint64_t seed;
  int step;
};
__device__ __forceinline__ uint32_t batch_row(const BatchDraw& d, int B, int b) {
  if (!d.draw) return (uint32_t)b;
  uint64_t z = d.seed + ((uint64_t)d.step * (uint64_t)B + (uint64_t)b + 1ull) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  // z mod n: the quotient from the reciprocal is at most two short
  uint64_t r = z - __umul64hi(z, d.recip) * d.n;
  if (r >= d.n) r -= d.n;
  if (r >= d.n) r -= d.n;
  return (uint32_t)r;
}

__device__ __forceinline__ float dot4(const float4& a, const float4& b, float s) {
  s += a.x * b.x;
  s += a.y * b.y;
  s += a.z * b.z;
  return s + a.w * b.w;
}
// sum over the workgroup's rows of a[row] b[row] (two LDS rows), in row order
__device__ __forceinline__ float dot_rows(const float* a, const float* b) {
  float s = 0.f;
#pragma unroll
  for (int r = 0; r < CHUNK; r += 4) s = dot4(*(const float4*)(a + r), *(const float4*)(b + r), s);
  return s;
}
__device__ __forceinline__ float sum_rows(const float* a) {
  float s = 0.f;
#pragma unroll
  for (int r = 0; r < CHUNK; ++r) s += a[r];
  return s;
}

// Forward and backward pass of CHUNK rows and their gradient sums (fixed
// order) into partial[block][MLP_PARAMS + 1], the squared error last.  Lane =
// row, wave w = hidden units 8 w .. 8 w + 7 of each layer, so that the weights
// are wave-uniform (scalar loads) and an LDS array [unit][row] is read without
// bank conflicts in the passes and 16 bytes at a time in the gradient sums.
__global__ __launch_bounds__(256) void k_mlp_batch(const float* __restrict__ P, const float* __restrict__ x,
                                                   const float* __restrict__ t, BatchDraw draw, int B,
                                                   float* __restrict__ partial) {
  __shared__ __align__(16) float sx[MLP_IN][ROWS];
  __shared__ __align__(16) float h1[MLP_HID][ROWS], h2[MLP_HID][ROWS], z1[MLP_HID][ROWS], z2[MLP_HID][ROWS];
  __shared__ __align__(16) float sy[4][ROWS], sdy[ROWS], ssq[ROWS];
  constexpr int U = MLP_HID / 4;  // units per wave
  const float* W1 = P;
  const float* b1 = W1 + MLP_IN * MLP_HID;
  const float* W2 = b1 + MLP_HID;
  const float* b2 = W2 + MLP_HID * MLP_HID;
  const float* W3 = b2 + MLP_HID;
  const int r = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), u0 = w * U;
  const int b = blockIdx.x * CHUNK + r;
  const bool live = b < B;  // rows past the batch repeat its last one with no error
  const size_t row = batch_row(draw, B, live ? b : B - 1);
  float xi[MLP_IN];
#pragma unroll
  for (int i = 0; i < MLP_IN; ++i) xi[i] = x[row * MLP_IN + i];
  const float target = t[row];
#pragma unroll
  for (int j = 0; j < U; ++j) {
    float z = b1[u0 + j];
#pragma unroll
    for (int i = 0; i < MLP_IN; ++i) z += xi[i] * W1[i * MLP_HID + u0 + j];
    h1[u0 + j][r] = tanhf(z);
  }
  if (w == 0) {
#pragma unroll
    for (int i = 0; i < MLP_IN; ++i) sx[i][r] = xi[i];
  }
  __syncthreads();
  float z[U];
#pragma unroll
  for (int j = 0; j < U; ++j) z[j] = b2[u0 + j];
#pragma unroll 8
  for (int h = 0; h < MLP_HID; ++h) {
    const float a = h1[h][r];
#pragma unroll
    for (int j = 0; j < U; ++j) z[j] += a * W2[h * MLP_HID + u0 + j];
  }
  float y = 0.f;
#pragma unroll
  for (int j = 0; j < U; ++j) {
    z[j] = tanhf(z[j]);
    h2[u0 + j][r] = z[j];
    y += z[j] * W3[u0 + j];
  }
  sy[w][r] = y;
  __syncthreads();
  const float err = live ? W3[MLP_HID] + ((sy[0][r] + sy[1][r]) + (sy[2][r] + sy[3][r])) - target : 0.f;
  const float dy = 2.f * err / (float)B;
  if (w == 0) {
    sdy[r] = dy;
    ssq[r] = err * err;
  }
#pragma unroll
  for (int j = 0; j < U; ++j) z2[u0 + j][r] = dy * W3[u0 + j] * (1.f - z[j] * z[j]);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < U; ++j) z[j] = 0.f;
#pragma unroll 8
  for (int g = 0; g < MLP_HID; ++g) {
    const float d = z2[g][r];
#pragma unroll
    for (int j = 0; j < U; ++j) z[j] += d * W2[(u0 + j) * MLP_HID + g];
  }
#pragma unroll
  for (int j = 0; j < U; ++j) {
    const float a = h1[u0 + j][r];
    z1[u0 + j][r] = z[j] * (1.f - a * a);
  }
  __syncthreads();
  float* out = partial + (size_t)blockIdx.x * (MLP_PARAMS + 1);
  // W2[h][g], a 2 x 2 tile per thread
  {
    const int h = 2 * (threadIdx.x >> 4), g = 2 * (threadIdx.x & 15);
    float s00 = 0.f, s01 = 0.f, s10 = 0.f, s11 = 0.f;
#pragma unroll 4
    for (int k = 0; k < CHUNK; k += 4) {
      const float4 a0 = *(const float4*)&h1[h][k], a1 = *(const float4*)&h1[h + 1][k];
      const float4 c0 = *(const float4*)&z2[g][k], c1 = *(const float4*)&z2[g + 1][k];
      s00 = dot4(a0, c0, s00);
      s01 = dot4(a0, c1, s01);
      s10 = dot4(a1, c0, s10);
      s11 = dot4(a1, c1, s11);
    }
    float* o = out + MLP_IN * MLP_HID + MLP_HID + h * MLP_HID + g;
    o[0] = s00;
    o[1] = s01;
    o[MLP_HID] = s10;
    o[MLP_HID + 1] = s11;
  }
  // W1[i][h], b1, b2, W3, b3, squared error
  constexpr int REST = MLP_IN * MLP_HID + 3 * MLP_HID + 2;
  for (int p = threadIdx.x; p < REST; p += 256) {
    int q = p;
    if (q < MLP_IN * MLP_HID) {
      out[q] = dot_rows(sx[q / MLP_HID], z1[q % MLP_HID]);
    } else if ((q -= MLP_IN * MLP_HID) < MLP_HID) {
      out[MLP_IN * MLP_HID + q] = sum_rows(z1[q]);
    } else if ((q -= MLP_HID) < MLP_HID) {
      out[MLP_IN * MLP_HID + MLP_HID + MLP_HID * MLP_HID + q] = sum_rows(z2[q]);
    } else if ((q -= MLP_HID) < MLP_HID) {
      out[MLP_PARAMS - 1 - MLP_HID + q] = dot_rows(h2[q], sdy);
    } else if (q == MLP_HID) {
      out[MLP_PARAMS - 1] = sum_rows(sdy);
    } else {
      out[MLP_PARAMS] = sum_rows(ssq);
    }
  }
}

// Sums of the blocks' partials, 64 parameters per workgroup and 16 interleaved
// runs of blocks per parameter, added in a fixed order; Adam update when
// lr > 0 (c1, c2: 1 - beta^step).
constexpr int ADAM_RUNS = 16;
__global__ __launch_bounds__(64 * ADAM_RUNS) void k_mlp_adam(const float* __restrict__ partial, int nblk,
                                                             float* __restrict__ P, float* __restrict__ m,
                                                             float* __restrict__ v, float* __restrict__ grad_out,
                                                             float lr, float c1, float c2,
                                                             float* __restrict__ loss_out, int B) {
  __shared__ float part[ADAM_RUNS][64];
  const int lane = threadIdx.x & 63, run = threadIdx.x >> 6;
  const int p = blockIdx.x * 64 + lane;
  float s = 0.f;
  if (p <= MLP_PARAMS) {
#pragma unroll 8
    for (int k = run; k < nblk; k += ADAM_RUNS) s += partial[(size_t)k * (MLP_PARAMS + 1) + p];
  }
  part[run][lane] = s;
  __syncthreads();
  if (run != 0 || p > MLP_PARAMS) return;
  float g = 0.f;
#pragma unroll
  for (int k = 0; k < ADAM_RUNS; ++k) g += part[k][lane];
  if (p == MLP_PARAMS) {
    if (loss_out) *loss_out = g / (float)B;
    return;
  }
  if (grad_out) grad_out[p] = g;
  if (lr > 0.f) {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float mm = b1 * m[p] + (1.f - b1) * g;
    const float vv = b2 * v[p] + (1.f - b2) * g * g;
    m[p] = mm;
    v[p] = vv;
    const float mh = mm / c1;
    const float vh = vv / c2;
    P[p] -= lr * mh / (sqrtf(vh) + eps);
  }
}

__global__ void k_standardise(const float* __restrict__ raw, float* __restrict__ x, uint32_t n,
                              const float* __restrict__ mean, const float* __restrict__ inv_std) {
  const uint64_t e = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= (uint64_t)n * MLP_IN) return;
  const int i = (int)(e % MLP_IN);
  x[e] = (raw[e] - mean[i]) * inv_std[i];
}

// Per-input sums of x and x^2 (FP64) of chunks of raw features.
__global__ __launch_bounds__(256) void k_feature_moments(const float* __restrict__ raw, uint32_t n,
                                                         double* __restrict__ part) {
  __shared__ double s1[256][MLP_IN];
  __shared__ double s2[256][MLP_IN];
  double a[MLP_IN] = {0}, q[MLP_IN] = {0};
  for (uint32_t c = blockIdx.x * 256u + threadIdx.x; c < n; c += gridDim.x * 256u)
    for (int i = 0; i < MLP_IN; ++i) {
      const double v = raw[(size_t)c * MLP_IN + i];
      a[i] += v;
      q[i] += v * v;
    }
  for (int i = 0; i < MLP_IN; ++i) {
    s1[threadIdx.x][i] = a[i];
    s2[threadIdx.x][i] = q[i];
  }
  __syncthreads();
  if (threadIdx.x < 2 * MLP_IN) {
    const int i = threadIdx.x % MLP_IN;
    const bool sq = threadIdx.x >= MLP_IN;
    double s = 0;
    for (int k = 0; k < 256; ++k) s += sq ? s2[k][i] : s1[k][i];
    part[(size_t)blockIdx.x * 2 * MLP_IN + threadIdx.x] = s;
  }
}

// ------------------------------------------------------------ inference
// Network output of raw feature rows (n x 9) with the matrix-core path of the
// step kernel; whole wavefronts run it, rows past n read row n - 1.
__global__ __launch_bounds__(256) void k_mlp_eval(const MlpNet* __restrict__ net, const float* __restrict__ raw,
                                                  uint32_t n, float* __restrict__ y) {
  __shared__ TanhTable tt;
  tanh_table_fill(tt);
  const uint32_t c = blockIdx.x * 256u + threadIdx.x;
  const uint32_t r = c < n ? c : n - 1u;
  float f[MLP_IN];
#pragma unroll
  for (int i = 0; i < MLP_IN; ++i) f[i] = raw[(size_t)r * MLP_IN + i];
  const float out = closure_wave(net, tt, f);
  if (c < n) y[c] = out;
}

// ------------------------------------------------------------ data
// Coarse cell (I, J, K) of an m^3 periodic coarse grid averages the fine
// cells r I .. r I + r - 1 (each axis) of the fine grid's unique n^3 region
// (the fine layout may carry duplicated x / y boundary layers: strides fx, fxy).
// A read of the fine fields: a workgroup takes a run of `cells` coarse cells
// along I, lane = fine cell along the row (cells r of them <= FILTER_LANES), each
// lane summing its r x r column of rows, so that the reads are whole lines and
// n m^2 lanes share them (a thread per coarse cell read 4 bytes per line and
// left the chip to 128 workgroups: 259 us for 256^3 filtered 8 times, 270 MB).
// The columns then add in fine x order, one (cell, quantity) per thread.
// Widths under FILTER_MIN gain nothing from it: a wave of k_les_filter_cells
// reads most of its lines there too, in one pass without LDS (us per call, cells
// / lanes: 256^3 by 1 223 / 360, by 2 125 / 141, 258^3 by 3 106 / 145, 256^3 by 4
// 118 / 77, 300^3 by 5 194 / 163, 256^3 by 8 254 / 61).
constexpr int FILTER_LANES = 256, FILTER_SUMS = 10, FILTER_MIN = 4;
__global__ __launch_bounds__(FILTER_LANES) void k_les_filter(const float* __restrict__ rho,
                                                             const float* __restrict__ ux,
                                                             const float* __restrict__ uy,
                                                             const float* __restrict__ uz, int fx, int fxy, int r,
                                                             int m, int cells, int runs, float* __restrict__ out) {
  __shared__ double col[FILTER_SUMS][FILTER_LANES];
  __shared__ double tot[FILTER_SUMS][FILTER_LANES];
  const uint32_t run = blockIdx.x % (uint32_t)runs, line = blockIdx.x / (uint32_t)runs;
  const int J = (int)(line % (uint32_t)m), K = (int)(line / (uint32_t)m);
  const int I0 = (int)run * cells, nc = min(cells, m - I0), lanes = nc * r;
  const int t = threadIdx.x;
  if (t < lanes) {
    double s[FILTER_SUMS] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int k = 0; k < r; ++k)
      for (int j = 0; j < r; ++j) {
        const size_t f = (size_t)(K * r + k) * fxy + (size_t)(J * r + j) * fx + ((size_t)I0 * r + t);
        const double d = rho[f], a = ux[f], b = uy[f], e = uz[f];
        s[0] += d;
        s[1] += d * a;
        s[2] += d * b;
        s[3] += d * e;
        s[4] += d * a * a;
        s[5] += d * b * b;
        s[6] += d * e * e;
        s[7] += d * a * b;
        s[8] += d * a * e;
        s[9] += d * b * e;
      }
#pragma unroll
    for (int c = 0; c < FILTER_SUMS; ++c) col[c][t] = s[c];
  }
  __syncthreads();
  for (int x = t; x < nc * FILTER_SUMS; x += FILTER_LANES) {
    const int cell = x % nc, c = x / nc;
    double s = 0;
    for (int i = 0; i < r; ++i) s += col[c][cell * r + i];
    tot[c][cell] = s;
  }
  __syncthreads();
  if (t >= nc) return;
  const uint32_t mc = (uint32_t)m * m * m;
  const size_t o = ((size_t)K * m + J) * m + I0 + t;
  const double inv = 1.0 / ((double)r * r * r);
  const double R = tot[0][t] * inv;
  const double U = tot[1][t] * inv / R, V = tot[2][t] * inv / R, W = tot[3][t] * inv / R;
  out[o] = (float)R;
  out[1 * (size_t)mc + o] = (float)U;
  out[2 * (size_t)mc + o] = (float)V;
  out[3 * (size_t)mc + o] = (float)W;
  out[4 * (size_t)mc + o] = (float)(tot[4][t] * inv / R - U * U);
  out[5 * (size_t)mc + o] = (float)(tot[5][t] * inv / R - V * V);
  out[6 * (size_t)mc + o] = (float)(tot[6][t] * inv / R - W * W);
  out[7 * (size_t)mc + o] = (float)(tot[7][t] * inv / R - U * V);
  out[8 * (size_t)mc + o] = (float)(tot[8][t] * inv / R - U * W);
  out[9 * (size_t)mc + o] = (float)(tot[9][t] * inv / R - V * W);
}

// The filter for widths under FILTER_MIN and above FILTER_LANES: a thread per
// coarse cell.
__global__ __launch_bounds__(256) void k_les_filter_cells(const float* __restrict__ rho, const float* __restrict__ ux,
                                                          const float* __restrict__ uy, const float* __restrict__ uz,
                                                          int fx, int fxy, int r, int m, float* __restrict__ out) {
  const uint32_t c = blockIdx.x * 256u + threadIdx.x;
  const uint32_t mc = (uint32_t)m * m * m;
  if (c >= mc) return;
  const int I = c % m, J = (c / m) % m, K = c / (m * m);
  double sr = 0, sx = 0, sy = 0, sz = 0, sxx = 0, syy = 0, szz = 0, sxy = 0, sxz = 0, syz = 0;
  for (int k = 0; k < r; ++k)
    for (int j = 0; j < r; ++j)
      for (int i = 0; i < r; ++i) {
        const size_t f = (size_t)(K * r + k) * fxy + (size_t)(J * r + j) * fx + (I * r + i);
        const double d = rho[f], a = ux[f], b = uy[f], e = uz[f];
        sr += d;
        sx += d * a;
        sy += d * b;
        sz += d * e;
        sxx += d * a * a;
        syy += d * b * b;
        szz += d * e * e;
        sxy += d * a * b;
        sxz += d * a * e;
        syz += d * b * e;
      }
  const double inv = 1.0 / (double)(r * r * r);
  const double R = sr * inv;
  const double U = sx * inv / R, V = sy * inv / R, W = sz * inv / R;
  float* o = out;
  o[0 * (size_t)mc + c] = (float)R;
  o[1 * (size_t)mc + c] = (float)U;
  o[2 * (size_t)mc + c] = (float)V;
  o[3 * (size_t)mc + c] = (float)W;
  o[4 * (size_t)mc + c] = (float)(sxx * inv / R - U * U);
  o[5 * (size_t)mc + c] = (float)(syy * inv / R - V * V);
  o[6 * (size_t)mc + c] = (float)(szz * inv / R - W * W);
  o[7 * (size_t)mc + c] = (float)(sxy * inv / R - U * V);
  o[8 * (size_t)mc + c] = (float)(sxz * inv / R - U * W);
  o[9 * (size_t)mc + c] = (float)(syz * inv / R - V * W);
}

__global__ __launch_bounds__(256) void k_les_targets(const float* __restrict__ co, int m, float nu,
                                                     float* __restrict__ feat, float* __restrict__ target) {
  const uint32_t c = blockIdx.x * 256u + threadIdx.x;
  const uint32_t mc = (uint32_t)m * m * m;
  if (c >= mc) return;
  const int I = c % m, J = (c / m) % m, K = c / (m * m);
  auto at = [&](int comp, int i, int j, int k) -> float {
    i = (i + m) % m;
    j = (j + m) % m;
    k = (k + m) % m;
    return co[(size_t)comp * mc + ((size_t)k * m + j) * m + i];
  };
  // g[a][b] = d_a u_b, central differences
  float g[3][3];
  for (int b = 0; b < 3; ++b) {
    g[0][b] = 0.5f * (at(1 + b, I + 1, J, K) - at(1 + b, I - 1, J, K));
    g[1][b] = 0.5f * (at(1 + b, I, J + 1, K) - at(1 + b, I, J - 1, K));
    g[2][b] = 0.5f * (at(1 + b, I, J, K + 1) - at(1 + b, I, J, K - 1));
  }
  const float S[6] = {g[0][0], g[1][1], g[2][2], 0.5f * (g[0][1] + g[1][0]), 0.5f * (g[0][2] + g[2][0]),
                      0.5f * (g[1][2] + g[2][1])};
  const float rho = co[c];
  const float t0 = co[4 * (size_t)mc + c], t1 = co[5 * (size_t)mc + c], t2 = co[6 * (size_t)mc + c];
  const float tr = (t0 + t1 + t2) / 3.f;
  const float dev[6] = {t0 - tr, t1 - tr, t2 - tr, co[7 * (size_t)mc + c], co[8 * (size_t)mc + c],
                        co[9 * (size_t)mc + c]};
  float num = 0.f, den = 0.f;
  for (int a = 0; a < 6; ++a) {
    const float w = a < 3 ? 1.f : 2.f;
    num += w * dev[a] * S[a];
    den += w * S[a] * S[a];
  }
  den *= 2.f;
  const float nut = den > 0.f ? fmaxf(0.f, -num / den) : 0.f;
  const float te = 3.f * (nu + nut) + 0.5f;
  const float k = -(2.f / 3.f) * rho * te;
  // central second moments kappa = Pi + rho/3 I
  float x[MLP_IN];
  closure_features(rho, k * S[0] + rho / 3.f, k * S[1] + rho / 3.f, k * S[2] + rho / 3.f, k * S[3], k * S[4],
                   k * S[5], x);
  for (int i = 0; i < MLP_IN; ++i) feat[(size_t)c * MLP_IN + i] = x[i];
  target[c] = nut / MLP_NU_SCALE;
}

// Host packing of a flat parameter vector into the device image.
static uint16_t bf16_bits(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  const uint32_t lsb = (u >> 16) & 1u;
  u += 0x7fffu + lsb;  // round to nearest even (finite inputs)
  return (uint16_t)(u >> 16);
}

void closure_pack(const float* p, const float* mean, const float* std_, MlpNet& net) {
  const float* W1 = p;
  const float* b1 = W1 + MLP_IN * MLP_HID;
  const float* W2 = b1 + MLP_HID;
  const float* b2 = W2 + MLP_HID * MLP_HID;
  const float* W3 = b2 + MLP_HID;
  memset(&net, 0, sizeof(net));
  for (int l = 0; l < 64; ++l) {
    const int half = l / 32, row = l % 32;
    for (int j = 0; j < 8; ++j) {
      const int k = 8 * half + j;
      net.a1[l][j] = bf16_bits(k < MLP_IN ? W1[k * MLP_HID + row] : 0.f);
      for (int s = 0; s < 2; ++s) net.a2[s][l][j] = bf16_bits(W2[acc_row(8 * s + j, half) * MLP_HID + row]);
    }
    for (int r = 0; r < 16; ++r) {
      const int h = acc_row(r, half);
      net.b1[l][r] = b1[h];
      net.b2[l][r] = b2[h];
      net.w3[l][r] = W3[h];
    }
  }
  net.b3 = W3[MLP_HID];
  for (int i = 0; i < MLP_IN; ++i) {
    net.mean[i] = mean[i];
    net.inv_std[i] = 1.f / std_[i];
  }
}

}  // namespace psl

using namespace psl;

struct psl_mlp {
  float params[MLP_PARAMS];
  float mean[MLP_IN];
  float std_[MLP_IN];
  MlpNet* d_net = nullptr;  // packed device image (inference)
};

const MlpNet* psl_mlp_device_net(const psl_mlp* m) { return m ? m->d_net : nullptr; }

namespace {

int upload_net(psl_mlp* m) {
  MlpNet net;
  closure_pack(m->params, m->mean, m->std_, net);
  PSL_HIP_TRY(hipMemcpy(m->d_net, &net, sizeof(net), hipMemcpyHostToDevice));
  return PSL_OK;
}

struct DevBuf {
  void* p = nullptr;
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
  int alloc(size_t bytes) {
    if (hipMalloc(&p, bytes) != hipSuccess) {
      set_error("hipMalloc failed in the closure trainer");
      return PSL_E_NOMEM;
    }
    return PSL_OK;
  }
  template <class T>
  T* as() const {
    return (T*)p;
  }
};

// One forward/backward over `B` rows and either an Adam step (lr > 0) or only
// the gradient; loss to *loss.
int train_pass(const float* x, const float* t, const BatchDraw& draw, int B, float* P, float* mo, float* ve,
               float* grad, float lr, int step, float* loss_dev, float* partial) {
  const int nblk = (B + CHUNK - 1) / CHUNK;
  k_mlp_batch<<<nblk, 256>>>(P, x, t, draw, B, partial);
  PSL_LAUNCH_CHECK();
  const float c1 = (float)(1.0 - std::pow((double)0.9f, step)), c2 = (float)(1.0 - std::pow((double)0.999f, step));
  k_mlp_adam<<<(MLP_PARAMS + 1 + 63) / 64, 64 * ADAM_RUNS>>>(partial, nblk, P, mo, ve, grad, lr, c1, c2, loss_dev, B);
  PSL_LAUNCH_CHECK();
  return PSL_OK;
}

size_t partial_bytes(int B) { return (size_t)((B + CHUNK - 1) / CHUNK) * (MLP_PARAMS + 1) * sizeof(float); }

}  // namespace

extern "C" {

int psl_mlp_create(psl_mlp** out) {
  PSL_CHECK_ARG(out, "null argument");
  psl_mlp* m = new psl_mlp();
  memset(m->params, 0, sizeof(m->params));
  for (int i = 0; i < MLP_IN; ++i) {
    m->mean[i] = 0.f;
    m->std_[i] = 1.f;
  }
  if (hipMalloc(&m->d_net, sizeof(MlpNet)) != hipSuccess) {
    delete m;
    set_error("hipMalloc of the network image failed");
    return PSL_E_NOMEM;
  }
  int rc = upload_net(m);
  if (rc) {
    (void)hipFree(m->d_net);
    delete m;
    return rc;
  }
  *out = m;
  return PSL_OK;
}

int psl_mlp_destroy(psl_mlp* m) {
  if (!m) return PSL_OK;
  (void)hipDeviceSynchronize();
  if (m->d_net) (void)hipFree(m->d_net);
  delete m;
  return PSL_OK;
}

int psl_mlp_set_params(psl_mlp* m, const float* params, const float* mean, const float* std_) {
  PSL_CHECK_ARG(m && params, "null argument");
  memcpy(m->params, params, sizeof(m->params));
  if (mean) memcpy(m->mean, mean, sizeof(m->mean));
  if (std_) {
    for (int i = 0; i < MLP_IN; ++i) PSL_CHECK_ARG(std_[i] > 0.f, "standard deviations must be positive");
    memcpy(m->std_, std_, sizeof(m->std_));
  }
  return upload_net(m);
}

int psl_mlp_get_params(const psl_mlp* m, float* params, float* mean, float* std_) {
  PSL_CHECK_ARG(m, "null network");
  if (params) memcpy(params, m->params, sizeof(m->params));
  if (mean) memcpy(mean, m->mean, sizeof(m->mean));
  if (std_) memcpy(std_, m->std_, sizeof(m->std_));
  return PSL_OK;
}

int psl_mlp_loss_grad(const psl_mlp* m, const float* x_dev, const float* t_dev, int n, double* loss, float* grad) {
  PSL_CHECK_ARG(m && x_dev && t_dev && n > 0, "bad arguments");
  DevBuf dpart, dP, dG, dL;
  int rc = dpart.alloc(partial_bytes(n));
  if (!rc) rc = dP.alloc(sizeof(m->params));
  if (!rc) rc = dG.alloc(sizeof(m->params));
  if (!rc) rc = dL.alloc(sizeof(float));
  if (rc) return rc;
  PSL_HIP_TRY(hipMemcpy(dP.p, m->params, sizeof(m->params), hipMemcpyHostToDevice));
  rc = train_pass(x_dev, t_dev, BatchDraw{}, n, dP.as<float>(), nullptr, nullptr, dG.as<float>(), 0.f, 1,
                  dL.as<float>(), dpart.as<float>());
  if (rc) return rc;
  float l = 0.f;
  PSL_HIP_TRY(hipMemcpy(&l, dL.p, sizeof(float), hipMemcpyDeviceToHost));
  if (loss) *loss = l;
  if (grad) PSL_HIP_TRY(hipMemcpy(grad, dG.p, sizeof(m->params), hipMemcpyDeviceToHost));
  return PSL_OK;
}

int psl_mlp_train(psl_mlp* m, const float* raw_dev, const float* t_dev, int n, int batch, int iters, float lr,
                  uint64_t seed, float* loss_hist) {
  PSL_CHECK_ARG(m && raw_dev && t_dev && n > 0 && batch > 0 && iters > 0 && lr > 0.f, "bad arguments");
  // standardisation from the data (FP64 moments)
  const int nblk_m = 256;
  DevBuf dpart, dx, dsum, dP, dm, dv, dloss, dmean, dinv;
  int rc = dpart.alloc((size_t)nblk_m * 2 * MLP_IN * sizeof(double));
  if (!rc) rc = dx.alloc((size_t)n * MLP_IN * sizeof(float));
  if (!rc) rc = dsum.alloc(partial_bytes(batch));
  if (!rc) rc = dP.alloc(sizeof(m->params));
  if (!rc) rc = dm.alloc(sizeof(m->params));
  if (!rc) rc = dv.alloc(sizeof(m->params));
  if (!rc) rc = dloss.alloc((size_t)iters * sizeof(float));
  if (!rc) rc = dmean.alloc(MLP_IN * sizeof(float));
  if (!rc) rc = dinv.alloc(MLP_IN * sizeof(float));
  if (rc) return rc;
  k_feature_moments<<<nblk_m, 256>>>(raw_dev, (uint32_t)n, dpart.as<double>());
  PSL_LAUNCH_CHECK();
  std::vector<double> part((size_t)nblk_m * 2 * MLP_IN);
  PSL_HIP_TRY(hipMemcpy(part.data(), dpart.p, part.size() * sizeof(double), hipMemcpyDeviceToHost));
  float inv[MLP_IN];
  for (int i = 0; i < MLP_IN; ++i) {
    double s = 0, q = 0;
    for (int k = 0; k < nblk_m; ++k) {
      s += part[(size_t)k * 2 * MLP_IN + i];
      q += part[(size_t)k * 2 * MLP_IN + MLP_IN + i];
    }
    const double mu = s / n, var = std::max(q / n - mu * mu, 0.0);
    m->mean[i] = (float)mu;
    m->std_[i] = (float)std::max(std::sqrt(var), 1e-6);
    inv[i] = 1.f / m->std_[i];
  }
  PSL_HIP_TRY(hipMemcpy(dmean.p, m->mean, sizeof(m->mean), hipMemcpyHostToDevice));
  PSL_HIP_TRY(hipMemcpy(dinv.p, inv, sizeof(inv), hipMemcpyHostToDevice));
  k_standardise<<<(uint32_t)(((uint64_t)n * MLP_IN + 255) / 256), 256>>>(raw_dev, dx.as<float>(), (uint32_t)n,
                                                                        dmean.as<float>(), dinv.as<float>());
  PSL_LAUNCH_CHECK();
  PSL_HIP_TRY(hipMemcpy(dP.p, m->params, sizeof(m->params), hipMemcpyHostToDevice));
  PSL_HIP_TRY(hipMemset(dm.p, 0, sizeof(m->params)));
  PSL_HIP_TRY(hipMemset(dv.p, 0, sizeof(m->params)));
  for (int it = 0; it < iters; ++it) {
    rc = train_pass(dx.as<float>(), t_dev, BatchDraw{true, (uint32_t)n, ~0ull / (uint64_t)n, seed, it}, batch,
                    dP.as<float>(), dm.as<float>(), dv.as<float>(), nullptr, lr, it + 1, dloss.as<float>() + it,
                    dsum.as<float>());
    if (rc) return rc;
  }
  PSL_HIP_TRY(hipMemcpy(m->params, dP.p, sizeof(m->params), hipMemcpyDeviceToHost));
  if (loss_hist) PSL_HIP_TRY(hipMemcpy(loss_hist, dloss.p, (size_t)iters * sizeof(float), hipMemcpyDeviceToHost));
  return upload_net(m);
}

int psl_mlp_eval(const psl_mlp* m, const float* raw_dev, int n, float* y_dev) {
  PSL_CHECK_ARG(m && raw_dev && y_dev && n > 0, "bad arguments");
  k_mlp_eval<<<(n + 255) / 256, 256>>>(m->d_net, raw_dev, (uint32_t)n, y_dev);
  PSL_LAUNCH_CHECK();
  PSL_HIP_TRY(hipDeviceSynchronize());
  return PSL_OK;
}

int psl_les_filter(const float* rho, const float* ux, const float* uy, const float* uz, int fine_nx, int fine_ny,
                   int n, int r, float* coarse) {
  PSL_CHECK_ARG(rho && ux && uy && uz && coarse, "null argument");
  PSL_CHECK_ARG(r > 0 && n > 0 && n % r == 0 && fine_nx >= n && fine_ny >= n, "bad filter geometry");
  const int m = n / r;
  const uint32_t mc = (uint32_t)m * m * m;
  if (r >= FILTER_MIN && r <= FILTER_LANES) {
    const int cells = std::min(m, FILTER_LANES / r), runs = (m + cells - 1) / cells;
    k_les_filter<<<(uint32_t)runs * m * m, FILTER_LANES>>>(rho, ux, uy, uz, fine_nx, fine_nx * fine_ny, r, m, cells,
                                                          runs, coarse);
  } else {
    k_les_filter_cells<<<(mc + 255) / 256, 256>>>(rho, ux, uy, uz, fine_nx, fine_nx * fine_ny, r, m, coarse);
  }
  PSL_LAUNCH_CHECK();
  PSL_HIP_TRY(hipDeviceSynchronize());
  return PSL_OK;
}

int psl_les_targets(const float* coarse, int m, float nu, float* feat, float* target) {
  PSL_CHECK_ARG(coarse && feat && target && m > 2, "bad arguments");
  const uint32_t mc = (uint32_t)m * m * m;
  k_les_targets<<<(mc + 255) / 256, 256>>>(coarse, m, nu, feat, target);
  PSL_LAUNCH_CHECK();
  PSL_HIP_TRY(hipDeviceSynchronize());
  return PSL_OK;
}

}  // extern "C"
