// Fused distance -> Gaussian kernel -> log-sum op and its backward helpers.
// The kernel is the one the Ferguson sweep sums, K_ij = exp(-D_ij / (2 eps))
// (fergusonE.py:36-43); the loss per eps is L = sum_i log sum_j K_ij.
#include "common.h"

namespace memi {

constexpr int EG = 8;  // eps values per block

// S[e][i] = sum_j K^e_ij, T[e][i] = sum_j K^e_ij D_ij; block = (row i, group of EG eps)
__global__ __launch_bounds__(256) void k_kernel_rowsums(const float* __restrict__ D, int n,
                                                        const double* __restrict__ eps,
                                                        int n_eps, double* __restrict__ S,
                                                        double* __restrict__ T) {
  __shared__ double red[8];
  const int i = blockIdx.x;
  const int e0 = blockIdx.y * EG;
  double c[EG], s[EG], t[EG];
#pragma unroll
  for (int q = 0; q < EG; ++q) {
    c[q] = (e0 + q < n_eps) ? 1.0 / (2.0 * eps[e0 + q]) : 0.0;
    s[q] = t[q] = 0.0;
  }
  const float* row = D + (int64_t)i * n;
  for (int j = threadIdx.x; j < n; j += blockDim.x) {
    const double d = row[j];
#pragma unroll
    for (int q = 0; q < EG; ++q) {
      const double k = exp(-d * c[q]);
      s[q] += k;
      t[q] += k * d;
    }
  }
#pragma unroll
  for (int q = 0; q < EG; ++q) {
    const double a = block_sum(s[q], red);
    const double b = block_sum(t[q], red);
    if (threadIdx.x == 0 && e0 + q < n_eps) {
      S[(int64_t)(e0 + q) * n + i] = a;
      T[(int64_t)(e0 + q) * n + i] = b;
    }
  }
}

// Wt[i][j] = sum_e g[e] (-1/(2 eps_e)) K^e_ij (1/S[e][i] + 1/S[e][j])   (K symmetric), and
// Wt[i][i] = 0: the i = j term of the gradient, w_k (X_ik C_ik^2 - C_ik C_ik X_ik) Wt_ii, is
// identically zero, while Wt_ii itself (K_ii = 1 at every eps, so the smallest eps dominates)
// can exceed the off-diagonal weights by 1e6 or more and would only feed rounding error of
// that size into the two float32 products Wt B and Wt Y, which cancel it in exact arithmetic.
//
// One 32 x 32 tile on or above the diagonal and its mirror image per block: entry (j, i) has the
// value of (i, j) wherever D is symmetric, so each exp serves both; the reciprocals of S and the
// constants of each eps are formed once per tile in LDS, not twice per entry.  Bound by the
// float64 exponentials.  n = 1000, 41 eps: 45 us, 112 for a thread per entry.
constexpr int GW = 32, GW_E = 16;   // tile side, eps per round
__global__ __launch_bounds__(256) void k_kernel_grad_weights(
    const float* __restrict__ D, int n, const double* __restrict__ eps, int n_eps,
    const double* __restrict__ S, const double* __restrict__ g, float* __restrict__ Wt) {
  const int bi = blockIdx.y, bj = blockIdx.x;
  if (bj < bi) return;
  __shared__ float dt[GW][GW + 1];
  __shared__ double ri[GW_E][GW], rj[GW_E][GW], ce[GW_E], ge[GW_E];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;      // column, row (mod 8) of the tile
  const int i0 = bi * GW, j0 = bj * GW;
  const int j = j0 + tx;
  // mirrored entries, transposed: dt[a][b] = D[j0 + a][i0 + b]
  for (int a = ty; a < GW; a += 8)
    dt[a][tx] = (j0 + a < n && i0 + tx < n) ? D[(int64_t)(j0 + a) * n + i0 + tx] : 0.f;
  float dv[4];
  double w[4] = {0.0, 0.0, 0.0, 0.0}, wm[4] = {0.0, 0.0, 0.0, 0.0};
  bool same = true;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int i = i0 + ty + 8 * u;
    dv[u] = (i < n && j < n) ? D[(int64_t)i * n + j] : 0.f;
    same = same && dv[u] == dt[tx][ty + 8 * u];
  }
  const bool mirror = __syncthreads_and(same);
  for (int q0 = 0; q0 < n_eps; q0 += GW_E) {
    __syncthreads();
    const int nq = min(GW_E, n_eps - q0);
    for (int x = threadIdx.x; x < nq * GW; x += 256) {
      const int q = x >> 5, a = x & 31;
      const double* Sq = S + (int64_t)(q0 + q) * n;
      ri[q][a] = i0 + a < n ? 1.0 / Sq[i0 + a] : 0.0;
      rj[q][a] = j0 + a < n ? 1.0 / Sq[j0 + a] : 0.0;
    }
    if ((int)threadIdx.x < nq) {
      ce[threadIdx.x] = 1.0 / (2.0 * eps[q0 + threadIdx.x]);
      ge[threadIdx.x] = g[q0 + threadIdx.x] * -ce[threadIdx.x];
    }
    __syncthreads();
    for (int q = 0; q < nq; ++q) {
      const double c = ce[q], gc = ge[q], r = rj[q][tx];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        w[u] += gc * exp(-(double)dv[u] * c) * (ri[q][ty + 8 * u] + r);
      if (!mirror) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
          wm[u] += gc * exp(-(double)dt[tx][ty + 8 * u] * c) * (ri[q][ty + 8 * u] + r);
      }
    }
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int i = i0 + ty + 8 * u;
    if (i < n && j < n) Wt[(int64_t)i * n + j] = i == j ? 0.f : (float)w[u];
  }
  if (bi == bj && mirror) return;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 4; ++u) dt[tx][ty + 8 * u] = (float)(mirror ? w[u] : wm[u]);
  __syncthreads();
  if (bi != bj)
    for (int a = ty; a < GW; a += 8)
      if (j0 + a < n && i0 + tx < n) Wt[(int64_t)(j0 + a) * n + i0 + tx] = dt[a][tx];
}

// The right operand of the backward product, row i = [C^2 | C Re X | C Im X] of image i over its Kh
// half-spectrum bins, and the gradient from the product's rows [WB | WYr | WYi]:
// out = 2 w_k (X WB - C (WYr + i WYi)), w_k the bin's half-spectrum weight.  One pass over memory
// each, which bounds them.  n = 1000, 128 x 128: 32 and 40 us; as separate elementwise
// operations the two took 385.
__global__ __launch_bounds__(256) void k_grad_operand(const float2* __restrict__ fy,
                                                      const float* __restrict__ ctf, int64_t n,
                                                      int64_t Kh, float* __restrict__ M) {
  const int64_t k = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (k >= Kh) return;
  for (int64_t i = blockIdx.y; i < n; i += gridDim.y) {
    const float C = ctf[i * Kh + k];
    const float2 X = fy[i * Kh + k];
    float* m = M + i * 3 * Kh + k;
    m[0] = C * C;
    m[Kh] = C * X.x;
    m[2 * Kh] = C * X.y;
  }
}

__global__ __launch_bounds__(256) void k_grad_combine(const float2* __restrict__ fy,
                                                      const float* __restrict__ ctf,
                                                      const float* __restrict__ WM, int64_t n,
                                                      int N, float2* __restrict__ out) {
  const int Nh = N / 2 + 1;
  const int64_t Kh = (int64_t)N * Nh;
  const int64_t k = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (k >= Kh) return;
  const float w2 = 2.f * half_weight((int)(k % Nh), N);
  for (int64_t i = blockIdx.y; i < n; i += gridDim.y) {
    const float C = ctf[i * Kh + k];
    const float2 X = fy[i * Kh + k];
    const float* m = WM + i * 3 * Kh + k;
    const float wb = m[0];
    out[i * Kh + k] =
        make_float2(w2 * (X.x * wb - C * m[Kh]), w2 * (X.y * wb - C * m[2 * Kh]));
  }
}

}  // namespace memi

using namespace memi;

extern "C" {

int memi_kernel_rowsums(const float* D, int n, const double* eps, int n_eps, double* S, double* T,
                        void* stream) {
  MEMI_CHECK_ARG(D && eps && S && T && n > 0 && n_eps > 0, "memi_kernel_rowsums: bad arguments");
  dim3 g((unsigned)n, (unsigned)((n_eps + EG - 1) / EG));
  hipLaunchKernelGGL(k_kernel_rowsums, g, dim3(256), 0, (hipStream_t)stream, D, n, eps, n_eps, S,
                     T);
  MEMI_CHECK_LAUNCH("k_kernel_rowsums");
  return MEMI_OK;
}

int memi_kernel_grad_weights(const float* D, int n, const double* eps, int n_eps, const double* S,
                             const double* g, float* Wt, void* stream) {
  MEMI_CHECK_ARG(D && eps && S && g && Wt && n > 0 && n_eps > 0,
                 "memi_kernel_grad_weights: bad arguments");
  const unsigned nb = (unsigned)((n + GW - 1) / GW);
  MEMI_CHECK_ARG(nb < 65536, "memi_kernel_grad_weights: n=%d too large", n);
  hipLaunchKernelGGL(k_kernel_grad_weights, dim3(nb, nb), dim3(256), 0, (hipStream_t)stream, D, n,
                     eps, n_eps, S, g, Wt);
  MEMI_CHECK_LAUNCH("k_kernel_grad_weights");
  return MEMI_OK;
}

int memi_grad_operand(const void* fy, const float* ctf_half, int64_t n, int N, float* M,
                      void* stream) {
  MEMI_CHECK_ARG(fy && ctf_half && M && n >= 0 && N > 0, "memi_grad_operand: bad arguments");
  if (n == 0) return MEMI_OK;
  const int64_t Kh = (int64_t)N * (N / 2 + 1);
  const dim3 g((unsigned)((Kh + 255) / 256), (unsigned)std::min<int64_t>(n, 65535));
  hipLaunchKernelGGL(k_grad_operand, g, dim3(256), 0, (hipStream_t)stream, (const float2*)fy,
                     ctf_half, n, Kh, M);
  MEMI_CHECK_LAUNCH("k_grad_operand");
  return MEMI_OK;
}

int memi_grad_combine(const void* fy, const float* ctf_half, const float* WM, int64_t n, int N,
                      void* out, void* stream) {
  MEMI_CHECK_ARG(fy && ctf_half && WM && out && n >= 0 && N > 0,
                 "memi_grad_combine: bad arguments");
  if (n == 0) return MEMI_OK;
  const int64_t Kh = (int64_t)N * (N / 2 + 1);
  const dim3 g((unsigned)((Kh + 255) / 256), (unsigned)std::min<int64_t>(n, 65535));
  hipLaunchKernelGGL(k_grad_combine, g, dim3(256), 0, (hipStream_t)stream, (const float2*)fy,
                     ctf_half, WM, n, N, (float2*)out);
  MEMI_CHECK_LAUNCH("k_grad_combine");
  return MEMI_OK;
}

}  // extern "C"
