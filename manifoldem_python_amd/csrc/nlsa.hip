// Stage 3 NLSA kernels.  Reference: NLSA.py:23-158, get_wiener.py:9-21, svdRF.py:9-35,
// L2_distance.py:8-41, psiAnalysisParS2.py:89-90.
#include "common.h"
#include <type_traits>

namespace memi {

// ---------------------------------------------------------------- delay embedding -------
// ConD[i][j] = sum_{c<C} D[ord[i+c]][ord[j+c]] (NLSA.py:31-34 after the psi sort of
// psiAnalysisParS2.py:89-90).  A 32x32 output tile needs the (32+C-1)^2 gathered block,
// staged once in LDS; the diagonal sums then run in increasing c like the reference loop.
constexpr int CT = 32;
constexpr int CMAX = 97;  // largest delay order the LDS block holds (32 + 96 = 128 rows)

template <typename T>
__global__ __launch_bounds__(256) void k_condist(const T* __restrict__ D,
                                                 const int64_t* __restrict__ ord, int n, int C,
                                                 double* __restrict__ ConD) {
  extern __shared__ double blk[];  // (CT+C-1)^2
  const int m = n - C;
  const int S = CT + C - 1;
  const int i0 = blockIdx.y * CT, j0 = blockIdx.x * CT;
  for (int e = threadIdx.x; e < S * S; e += blockDim.x) {
    const int r = e / S, c = e % S;
    const int gi = i0 + r, gj = j0 + c;
    double v = 0.0;
    if (gi < n && gj < n) v = (double)D[ord[gi] * (int64_t)n + ord[gj]];
    blk[e] = v;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < CT * CT; e += blockDim.x) {
    const int r = e / CT, c = e % CT;
    const int i = i0 + r, j = j0 + c;
    if (i >= m || j >= m) continue;
    double s = 0.0;
    for (int k = 0; k < C; ++k) s += blk[(r + k) * S + (c + k)];
    ConD[(int64_t)i * m + j] = s;
  }
}

// ------------------------------------------------------------ supervector spectra -------
// out[ii][c][k] = sum_{i<m} mu_psi[i][c] * spec[j][k] C[j][k] / W_i[k], j = C-1-ii+i,
// W_i[k] = sum_{t=i+1}^{i+C} C[t][k]^2 + 1/snr.
//
// A wave takes SG delays and four of the ell weights of 64 frequencies: 8 SG float32 sums per
// lane.  The waves of a workgroup hold the other delays and weights of the same frequencies and
// share the weights u[i][c] = mu_psi[i][c] / W_i (float64, rounded once), which they compute in
// turn, SG steps ahead, into LDS.  The spectra slide by one image per step; SG steps are unrolled
// so that every G sits in a register of its own.  With few frequencies a wave takes 2^kshift of
// them and cuts the steps into 64 >> kshift pieces, summed across its lanes at the end.
//
// Bound: float32 multiply-add issue (8 SG per step against ~25 other instructions) at two waves
// per SIMD, and 203 workgroups on 256 CUs: 1500 images of 160 x 160, 50 delays, 8 weights take
// 0.75 ms (40 TFLOP/s); 1.63 ms with 5 delays x 8 weights per thread, where each thread formed
// its own eight weights with a float64 division every 80 sums and waited for each step's loads.
constexpr int ELLMAX = 8;

template <int SG, typename OFF>
__global__ __launch_bounds__(512) void k_supervectors(
    const float2* __restrict__ spec, const float* __restrict__ ctf, int n, int64_t Kh, int C,
    const double* __restrict__ mu_psi, int ell, double snr, int kshift, int steps, int gpb,
    int halves, float2* __restrict__ out) {
  __shared__ float4 us[2][SG][2][64];        // the weights of two rounds of SG steps
  __shared__ double ws[SG][64];
  __shared__ double mus[2][SG * ELLMAX * 16];  // mu_psi of two rounds: [step][c][piece]
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = blockDim.x >> 6;
  const int half = w % halves;
  const int g0 = ((int)blockIdx.y * gpb + w / halves) * SG;     // this wave's first delay
  const int64_t k = ((int64_t)blockIdx.x << kshift) + (lane & ((1 << kshift) - 1));
  const int64_t kc = min(k, Kh - 1);
  const int m = n - C;
  const int i0 = (lane >> kshift) * steps;                       // this lane's steps
  // element offsets (OFF: 32 bits when they fit, one register per address); images outside the
  // steps' range are read at its ends and enter no sum
  auto img = [&](int j) { return (OFF)min(max(j, 0), n - 2) * (OFF)Kh + (OFF)kc; };
  auto ctf_at = [&](int t) { return ctf[(OFF)min(t, n - 1) * (OFF)Kh + (OFF)kc]; };
  double W = 1.0 / snr;
  for (int t = 1; t <= C; ++t) {
    const double c = ctf_at(i0 + t);
    W += c * c;
  }
  // mu_psi of steps c0 .. c0 + SG - 1 into LDS, zero past a piece's end
  const int pieces = 64 >> kshift;
  auto stage_mu = [&](int c0, double* to) {
#pragma unroll 1
    for (int e = threadIdx.x; e < SG * ell * pieces; e += blockDim.x) {
      const int q = e / (SG * ell), r = e % (SG * ell);
      const int st = c0 + r / ell, i = q * steps + st;
      to[r * pieces + q] = (st < steps && i < m) ? mu_psi[(int64_t)i * ell + r % ell] : 0.0;
    }
  };
  // the CTFs that leave and enter the window over steps c0 .. c0 + SG - 1
  float wa[SG], wb[SG];
  auto window = [&](int c0) {
#pragma unroll
    for (int t = 0; t < SG; ++t) {
      wa[t] = ctf_at(i0 + c0 + t + 1);
      wb[t] = ctf_at(i0 + c0 + t + 1 + C);
    }
  };
  // The weights of those steps: wave w computes every nw-th of them.  Every wave runs the window
  // sum through all steps and keeps its own ones in LDS (nobody else reads them), so that the
  // divisions stay out of the unrolled code, where they cost registers.
  auto weights = [&](float4(*u)[2][64], const double* mu) {
#pragma unroll
    for (int t = 0; t < SG; ++t) {
      if (t % nw == w) ws[t][lane] = W;
      const double a = wa[t], b = wb[t];
      W += b * b - a * a;
    }
#pragma unroll 1
    for (int t = w; t < SG; t += nw) {
      const double invW = 1.0 / ws[t][lane];
      const double* mp = mu + t * ell * pieces + (lane >> kshift);
#pragma unroll 1
      for (int h = 0; h < halves; ++h) {
        float v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c)
          v[c] = 4 * h + c < ell ? (float)(mp[(4 * h + c) * pieces] * invW) : 0.f;
        u[t][h][lane] = make_float4(v[0], v[1], v[2], v[3]);
      }
    }
  };
  float2 prev[SG], cur[SG], nx[SG];
  float nc[SG];
  const int j0 = C - 1 - g0 + i0;            // newest image of delay g0 at the first step
#pragma unroll
  for (int t = 0; t < SG; ++t) {
    const OFF a = img(j0 - SG + t), b = img(j0 + t);
    const float2 x = spec[a], y = spec[b];
    const float cx = ctf[a], cy = ctf[b];
    prev[t] = make_float2(x.x * cx, x.y * cx);
    cur[t] = make_float2(y.x * cy, y.y * cy);
  }
  float acc[SG][4][2];
#pragma unroll
  for (int d = 0; d < SG; ++d)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[d][c][0] = acc[d][c][1] = 0.f;
  stage_mu(0, mus[0]);
  stage_mu(SG, mus[1]);
  window(0);
  __syncthreads();
  weights(us[0], mus[0]);
  // Steps past a piece's end take zero for the images too: their weights are zero, but the history
  // holds images of other delays' sums, which need not be finite.  Only the rounds that reach past
  // an end (TAIL) pay for it.
  const int lim = min(steps, m - i0);
  const int full = min(steps, m - (pieces - 1) * steps);
  int b = 0;
  auto round = [&](auto TAIL, int c0) __attribute__((always_inline)) {
    __syncthreads();       // this round's weights are in us[b], the next one's mu in mus[b ^ 1]
    stage_mu(c0 + 2 * SG, mus[b]);
    if (g0 >= C) window(c0 + SG);            // a wave with no delays left only computes weights
    else {
#pragma unroll
      for (int t = 0; t < SG; ++t) {
        const OFF a = img(j0 + c0 + SG + t);
        nx[t] = spec[a];
        nc[t] = ctf[a];
      }
      float4 un = us[b][0][half][lane];
#pragma unroll
      for (int t = 0; t < SG; ++t) {
        const float4 u = un;
        if (t + 1 < SG) un = us[b][t + 1][half][lane];
#pragma unroll
        for (int d = 0; d < SG; ++d) {
          float2 g = t >= d ? cur[t >= d ? t - d : 0] : prev[t >= d ? 0 : SG + t - d];
          if (decltype(TAIL)::value && c0 + t >= lim) g = make_float2(0.f, 0.f);
          acc[d][0][0] += u.x * g.x;
          acc[d][0][1] += u.x * g.y;
          acc[d][1][0] += u.y * g.x;
          acc[d][1][1] += u.y * g.y;
          acc[d][2][0] += u.z * g.x;
          acc[d][2][1] += u.z * g.y;
          acc[d][3][0] += u.w * g.x;
          acc[d][3][1] += u.w * g.y;
        }
        // loads in flight across the second half, whose history needs fewer registers
        if (t == SG / 2) window(c0 + SG);
      }
#pragma unroll
      for (int t = 0; t < SG; ++t) {
        prev[t] = cur[t];
        cur[t] = make_float2(nx[t].x * nc[t], nx[t].y * nc[t]);
      }
    }
    b ^= 1;
    if (c0 + SG < steps) weights(us[b], mus[b]);
  };
  int c0 = 0;
  for (; c0 + SG <= full; c0 += SG) round(std::false_type{}, c0);
  for (; c0 < steps; c0 += SG) round(std::true_type{}, c0);
  for (int off = 1 << kshift; off < 64; off <<= 1)
#pragma unroll
    for (int d = 0; d < SG; ++d)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        acc[d][c][0] += __shfl_xor(acc[d][c][0], off, 64);
        acc[d][c][1] += __shfl_xor(acc[d][c][1], off, 64);
      }
  if ((lane >> kshift) != 0 || k >= Kh) return;
#pragma unroll
  for (int d = 0; d < SG; ++d)
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (g0 + d < C && 4 * half + c < ell)
        out[((int64_t)(g0 + d) * ell + 4 * half + c) * Kh + k] =
            make_float2(acc[d][c][0], acc[d][c][1]);
}

// ------------------------------------------------------------- tall-skinny algebra -------
constexpr int TGMAX = 8;

__global__ __launch_bounds__(256) void k_tall_gram(const double* __restrict__ A, int64_t M, int c,
                                                   double* __restrict__ G) {
  __shared__ double red[TGMAX * TGMAX][4];
  double s[TGMAX * (TGMAX + 1) / 2];
#pragma unroll
  for (int q = 0; q < TGMAX * (TGMAX + 1) / 2; ++q) s[q] = 0.0;
  for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < M;
       r += (int64_t)gridDim.x * blockDim.x) {
    double a[TGMAX];
#pragma unroll
    for (int x = 0; x < TGMAX; ++x) a[x] = (x < c) ? A[r * c + x] : 0.0;
    int q = 0;
#pragma unroll
    for (int x = 0; x < TGMAX; ++x)
#pragma unroll
      for (int y = x; y < TGMAX; ++y) s[q++] += a[x] * a[y];
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int q = 0;
#pragma unroll
  for (int x = 0; x < TGMAX; ++x)
#pragma unroll
    for (int y = x; y < TGMAX; ++y) {
      double v = s[q++];
      for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
      if (lane == 0) red[x * TGMAX + y][wid] = v;
    }
  __syncthreads();
  for (int e = threadIdx.x; e < c * c; e += blockDim.x) {
    const int x = e / c, y = e % c;
    const int xx = min(x, y), yy = max(x, y);
    const double v = red[xx * TGMAX + yy][0] + red[xx * TGMAX + yy][1] +
                     red[xx * TGMAX + yy][2] + red[xx * TGMAX + yy][3];
    atomicAdd(&G[e], v);
  }
}

struct SmallMat {
  double v[TGMAX * TGMAX];
};

__global__ void k_tall_apply(const double* __restrict__ A, int64_t M, int c, SmallMat B, int d,
                             double* __restrict__ Y) {
  for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < M;
       r += (int64_t)gridDim.x * blockDim.x) {
    double a[TGMAX];
    for (int x = 0; x < c; ++x) a[x] = A[r * c + x];
    for (int y = 0; y < d; ++y) {
      double s = 0.0;
      for (int x = 0; x < c; ++x) s += a[x] * B.v[x * d + y];
      Y[r * d + y] = s;
    }
  }
}

// column means of U2 [npix][q] (accumulated into mean[q]), then centre in place
__global__ void k_col_sum(const double* __restrict__ U, int64_t npix, int q,
                          double* __restrict__ colsum) {
  const int col = blockIdx.y * blockDim.x + threadIdx.x;
  if (col >= q) return;
  double s = 0.0;
#pragma unroll 8
  for (int64_t p = blockIdx.x; p < npix; p += gridDim.x) s += U[p * q + col];
  atomicAdd(&colsum[col], s);
}

__global__ void k_col_center(double* __restrict__ U, int64_t npix, int q,
                             const double* __restrict__ colsum) {
  const int64_t total = npix * q;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x)
    U[e] -= colsum[e % q] / (double)npix;
}

// G[a][b] += sum_p U[p][a] U[p][b] over a wave's pixel range, on v_mfma_f64_16x16x4_f64: one 16x16
// tile (a0 <= b0) of G per wave, four pixels per instruction straight from memory (a lane reads
// U[p + l / 16][a0 + l % 16], whole 128-byte lines), eight instructions' loads in flight.  Every
// tile below the diagonal is its mirror's transpose.  Bound: memory latency (npix = 25600,
// q = 100: 32 us; 100 us with both operands through LDS on the vector units).
typedef double doublex4_t __attribute__((ext_vector_type(4)));
constexpr int GC_ROWS = 512;               // pixels per wave

__global__ __launch_bounds__(256) void k_gram_cols(const double* __restrict__ U, int64_t npix,
                                                   int q, double* __restrict__ G) {
  if (blockIdx.y < blockIdx.x) return;
  const int a0 = blockIdx.x * 16, b0 = blockIdx.y * 16;
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int64_t p0 = ((int64_t)blockIdx.z * 4 + (threadIdx.x >> 6)) * GC_ROWS;
  const int64_t p1 = min(npix, p0 + GC_ROWS);
  const bool ina = a0 + lr < q, inb = b0 + lr < q;
  const double* ua = U + (ina ? a0 + lr : 0);
  const double* ub = U + (inb ? b0 + lr : 0);
  doublex4_t acc = {};
  for (int64_t pb = p0; pb < p1; pb += 32) {
    double a[8], b[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int64_t p = pb + 4 * e + lk;
      const bool in = p < p1;
      const int64_t at = (in ? p : p0) * q;
      a[e] = in && ina ? ua[at] : 0.0;
      b[e] = in && inb ? ub[at] : 0.0;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[e], b[e], acc, 0, 0, 0);
  }
  if (p0 >= npix || !inb) return;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int i = a0 + lk + 4 * e, j = b0 + lr;
    if (i >= q) continue;
    atomicAdd(&G[i * q + j], acc[e]);
    if (a0 != b0) atomicAdd(&G[j * q + i], acc[e]);
  }
}

// IMGT[p][j] = inv_sd[j] * sum_q Ubar[p][q] H[q][j] on v_mfma_f64_16x16x4_f64: 64 x 128 outputs
// per workgroup, 32 x 64 per wave (8 blocks of 16 x 16), K in pieces of 20 through LDS.  Lane l
// of an MFMA holds A[l % 16][l / 16], B[l / 16][l % 16] and rows l / 16 + 4 r of column l % 16 of
// the result.
//
// Bound: the float64 MFMAs and writing IMGT (npix = 25600, q = 100, 1400 columns: 98 us at the
// rate a large float64 product reaches, 58 us at a large copy's): 227 us, with the next piece's
// loads in flight during the products and two workgroups per CU (three without the prefetch: 280
// us; 128 x 128 outputs, one workgroup per CU: 454; the vector units with 4 x 4 outputs per
// thread, two LDS reads for every two products: 410).
constexpr int IM_P = 64, IM_J = 128, IM_K = 20;

__global__ __launch_bounds__(256, 2) void k_imgt(const double* __restrict__ U,
                                                 const double* __restrict__ H,
                                                 const double* __restrict__ inv_sd, int64_t npix,
                                                 int q, int ncols, double* __restrict__ out) {
  __shared__ double us2[2][IM_K][IM_P + 2], hs2[2][IM_K][IM_J + 2];
  const int64_t p0 = (int64_t)blockIdx.y * IM_P;
  const int j0 = blockIdx.x * IM_J;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int pw = (wv >> 1) * 32, jw = (wv & 1) * 64;            // this wave's corner
  const int lr = lane & 15, lk = lane >> 4;
  doublex4_t acc[2][4] = {};
  constexpr int NU = IM_P * IM_K / 256, NH = IM_J * IM_K / 256;
  double ru[NU], rh[NH];                     // the next piece, loaded during this one's products
  auto load = [&](int k0) {
#pragma unroll
    for (int e = 0; e < NU; ++e) {
      const int f = threadIdx.x + 256 * e, pr = f / IM_K, pk = k0 + f % IM_K;   // along U's rows
      ru[e] = (p0 + pr < npix && pk < q) ? U[(p0 + pr) * q + pk] : 0.0;
    }
#pragma unroll
    for (int e = 0; e < NH; ++e) {
      const int f = threadIdx.x + 256 * e, hk = k0 + f / IM_J, hj = j0 + f % IM_J;  // along H's
      rh[e] = (hj < ncols && hk < q) ? H[(int64_t)hk * ncols + hj] : 0.0;
    }
  };
  auto store = [&](int b) {
#pragma unroll
    for (int e = 0; e < NU; ++e) {
      const int f = threadIdx.x + 256 * e;
      us2[b][f % IM_K][f / IM_K] = ru[e];
    }
#pragma unroll
    for (int e = 0; e < NH; ++e) {
      const int f = threadIdx.x + 256 * e;
      hs2[b][f / IM_J][f % IM_J] = rh[e];
    }
  };
  load(0);
  store(0);
  __syncthreads();
  int bf = 0;
  for (int k0 = 0; k0 < q; k0 += IM_K, bf ^= 1) {
    double(*us)[IM_P + 2] = us2[bf];
    double(*hs)[IM_J + 2] = hs2[bf];
    load(k0 + IM_K);
#pragma unroll
    for (int k = 0; k < IM_K; k += 4) {
      double a[2], b[4];
#pragma unroll
      for (int r = 0; r < 2; ++r) a[r] = us[k + lk][pw + 16 * r + lr];
#pragma unroll
      for (int c = 0; c < 4; ++c) b[c] = hs[k + lk][jw + 16 * c + lr];
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          acc[r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[r], b[c], acc[r][c], 0, 0, 0);
    }
    store(bf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int j = j0 + jw + 16 * c + lr;
    if (j >= ncols) continue;
    const double sd = inv_sd[j];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t p = p0 + pw + 16 * r + lk + 4 * e;
        if (p < npix) out[p * ncols + j] = acc[r][c][e] * sd;
      }
  }
}

// ---------------------------------------------------------- reconstruction distances ----
// T[a][j] = sum_b Gq[a][b] H[b][j]   (Gq [q][q], H [q][ncols]).  One output per thread; eight
// terms' loads go out together (one at a time: 41 us instead of 11 for q = 100, 1400 columns).
__global__ void k_gq_h(const double* __restrict__ Gq, const double* __restrict__ H, int q,
                       int ncols, double* __restrict__ T) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  const int a = blockIdx.y;
  if (j >= ncols) return;
  double s = 0.0;
#pragma unroll 8
  for (int b = 0; b < q; ++b) s = fma(Gq[a * q + b], H[(int64_t)b * ncols + j], s);
  T[(int64_t)a * ncols + j] = s;
}

// Gram_jj = sum_a H[a][j] T[a][j] in increasing a with fma, the order k_recon_dist's tiles use,
// so its diagonal entries equal these bit for bit; inv_sd_j = 1 / sqrt(Gram_jj / npix).
__global__ void k_recon_diag(const double* __restrict__ H, const double* __restrict__ T, int q,
                             int ncols, double npix, double* __restrict__ dg,
                             double* __restrict__ inv_sd) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= ncols) return;
  double s = 0.0;
#pragma unroll 8
  for (int a = 0; a < q; ++a) s = fma(H[(int64_t)a * ncols + j], T[(int64_t)a * ncols + j], s);
  dg[j] = s;
  inv_sd[j] = 1.0 / sqrt(s / npix);
}

// 64x64 tiles of Gram = H^T T with the L2_distance epilogue of NLSA.py:141-146:
// C_ij = Gram_ij (inv_i inv_j), d = (C_ii + C_jj) - 2 C_ij, d < 1e-8 -> 0, out = sqrt(d)^2.
__global__ __launch_bounds__(256) void k_recon_dist(const double* __restrict__ H,
                                                    const double* __restrict__ T,
                                                    const double* __restrict__ dg,
                                                    const double* __restrict__ inv_sd, int q,
                                                    int ncols, float* __restrict__ out) {
  __shared__ double hs[16][65], ts[16][65];
  const int i0 = blockIdx.y * 64, j0 = blockIdx.x * 64;
  const int tr = threadIdx.x >> 4, tc = threadIdx.x & 15;
  double acc[4][4] = {};
  for (int k0 = 0; k0 < q; k0 += 16) {
    for (int e = threadIdx.x; e < 16 * 64; e += blockDim.x) {
      const int kk = e / 64, x = e % 64;
      const bool kin = k0 + kk < q;
      hs[kk][x] = (kin && i0 + x < ncols) ? H[(int64_t)(k0 + kk) * ncols + i0 + x] : 0.0;
      ts[kk][x] = (kin && j0 + x < ncols) ? T[(int64_t)(k0 + kk) * ncols + j0 + x] : 0.0;
    }
    __syncthreads();
    const int kend = min(16, q - k0);
    for (int kk = 0; kk < kend; ++kk) {
      double a[4], b[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        a[x] = hs[kk][tr * 4 + x];
        b[x] = ts[kk][tc * 4 + x];
      }
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) acc[x][y] = fma(a[x], b[y], acc[x][y]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int i = i0 + tr * 4 + x;
    if (i >= ncols) continue;
    const double ii = inv_sd[i];
    const double aai = dg[i] * (ii * ii);
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      const int j = j0 + tc * 4 + y;
      if (j >= ncols) continue;
      const double ij = inv_sd[j];
      const double c = acc[x][y] * (ii * ij);
      double d = (aai + dg[j] * (ij * ij)) - 2.0 * c;
      if (d < 1e-8) d = 0.0;
      const double r = sqrt(d);
      out[(int64_t)i * ncols + j] = (float)(r * r);
    }
  }
}

// ------------------------------------------------------------- 1-D open-manifold fit ----
// tau update of fit_1D_open_manifold_3D.py:64-160: for a point x and curve (a, b),
// R(tau) = sum_j (x_j - b_j - a_j cos(j pi tau))^2 (R_p.py:41-49) is stationary in (0, 1)
// where beta = cos(pi tau) is a root of the quintic of solve_d_R_d_tau_p_3D.py:35-60; tau is
// the candidate arccos(beta)/pi (real beta in [-1, 1]) or 0 or 1 of least R, first in order on
// ties.  The reference takes the roots from np.roots (a LAPACK eigensolve of the companion
// matrix) and keeps those with zero imaginary part.  Here the real roots come from monotone
// segments: the roots of p^(k) bracket those of p^(k-1), so isolating from the linear fourth
// derivative up gives every real root of p in [-1.01, 1.01] by safeguarded Newton steps.
// Where LAPACK's real/complex decision or the arg min is within rounding of a tie (a stationary
// value of p within 1e-10 of its scale: a near-double root; p(+-1) that small: a root at the
// edge; two candidates with R equal to 1e-12 of its scale; a zero leading or trailing
// coefficient, which np.roots treats specially) the point is flagged for the host to re-solve.
constexpr int FIT_BLOCK = 256;
constexpr double FIT_LO = -1.01, FIT_HI = 1.01;
constexpr double FIT_EPS = 2.220446049250313e-16;   // double precision unit roundoff x 2

struct FitCurve {
  double a[3], b[3];
};

__device__ inline double peval(const double* e, int d, double x) {
  double r = e[d];
  for (int k = d - 1; k >= 0; --k) r = fma(r, x, e[k]);
  return r;
}

// root of e (degree d) in the bracket [u, v] where e(u), e(v) have opposite signs and e is
// monotone; de is its derivative (degree d - 1)
__device__ double monotone_root(const double* e, int d, const double* de, double u, double v,
                                double pu) {
  double x = 0.5 * (u + v);
  for (int it = 0; it < 200; ++it) {
    const double px = peval(e, d, x);
    if (px == 0.0) return x;
    if ((px < 0.0) == (pu < 0.0)) {
      u = x;
      pu = px;
    } else {
      v = x;
    }
    if (v - u <= 4.0 * FIT_EPS * fmax(fabs(u), fabs(v)) || v - u <= 1e-300) break;
    const double dx = peval(de, d - 1, x);
    if (dx != 0.0) {
      const double step = px / dx;
      // a Newton step of a few ulps: x is the root to rounding (further steps only bounce
      // between the bracket's ends while bisection halves it to the last bit)
      if (fabs(step) <= 16.0 * FIT_EPS * fabs(x)) {
        const double xn = x - step;
        return (xn > u && xn < v) ? xn : x;
      }
    }
    double xn = dx != 0.0 ? x - px / dx : u;
    if (!(xn > u && xn < v)) xn = 0.5 * (u + v);
    if (xn == x) break;
    x = xn;
  }
  return x;
}

// real roots of e (degree d) in [FIT_LO, FIT_HI], ascending, given the ascending roots cr[0..nc)
// of its derivative strictly inside the interval
__device__ int segment_roots(const double* e, int d, const double* de, const double* cr, int nc,
                             double* out) {
  int n = 0;
  double u = FIT_LO, pu = peval(e, d, u);
  if (pu == 0.0) out[n++] = u;
  for (int s = 0; s <= nc; ++s) {
    const double v = s < nc ? cr[s] : FIT_HI;
    const double pv = peval(e, d, v);
    if (pv == 0.0) {
      if (n == 0 || out[n - 1] != v) out[n++] = v;
    } else if (pu != 0.0 && ((pu < 0.0) != (pv < 0.0))) {
      out[n++] = monotone_root(e, d, de, u, v, pu);
    }
    u = v;
    pu = pv;
  }
  return n;
}

__device__ inline int interior(const double* r, int n, double* out) {
  int m = 0;
  for (int i = 0; i < n; ++i)
    if (r[i] > FIT_LO && r[i] < FIT_HI) out[m++] = r[i];
  return m;
}

__device__ inline double fit_residual(const double x[3], const FitCurve& c, double tau) {
  double r = 0.0;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const double e = x[j] - c.b[j] - c.a[j] * cos(tau * (double)(j + 1) * M_PI);
    r += e * e;
  }
  return r;
}

__global__ __launch_bounds__(FIT_BLOCK) void k_fit1d_tau(const double* __restrict__ X, int n,
                                                         FitCurve c, double* __restrict__ tau,
                                                         int32_t* __restrict__ flag,
                                                         double* __restrict__ part) {
  __shared__ double red[13][FIT_BLOCK];
  const int i = blockIdx.x * FIT_BLOCK + threadIdx.x;
  double acc[13];
#pragma unroll
  for (int k = 0; k < 13; ++k) acc[k] = 0.0;
  if (i < n) {
    const double x[3] = {X[i * 3], X[i * 3 + 1], X[i * 3 + 2]};
    // np.roots order c0..c5 (solve_d_R_d_tau_p_3D.py:35-60), stored ascending: e[k] = c_{5-k}
    double e[6];
    e[5] = 48.0 * c.a[2] * c.a[2];
    e[4] = 0.0;
    e[3] = 8.0 * c.a[1] * c.a[1] - 48.0 * c.a[2] * c.a[2];
    e[2] = -12.0 * c.a[2] * (x[2] - c.b[2]);
    e[1] = c.a[0] * c.a[0] - 4.0 * c.a[1] * c.a[1] + 9.0 * c.a[2] * c.a[2] -
           4.0 * c.a[1] * (x[1] - c.b[1]);
    e[0] = -c.a[0] * (x[0] - c.b[0]) + 3.0 * c.a[2] * (x[2] - c.b[2]);
    int amb = (e[5] == 0.0 || e[0] == 0.0) ? 1 : 0;
    double t_best = 0.0;
    if (!amb) {
      // derivatives, each ascending
      double d1[5], d2[4], d3[3], d4[2];
      for (int k = 0; k < 5; ++k) d1[k] = (k + 1) * e[k + 1];
      for (int k = 0; k < 4; ++k) d2[k] = (k + 1) * d1[k + 1];
      for (int k = 0; k < 3; ++k) d3[k] = (k + 1) * d2[k + 1];
      for (int k = 0; k < 2; ++k) d4[k] = (k + 1) * d3[k + 1];
      double r4[1], r3[3], r2[4], r1[5], r0[6], tmp[6];
      int n4 = 0;
      {
        const double z = -d4[0] / d4[1];
        if (z > FIT_LO && z < FIT_HI) r4[n4++] = z;
      }
      int n3 = interior(tmp, segment_roots(d3, 2, d4, r4, n4, tmp), r3);
      int n2 = interior(tmp, segment_roots(d2, 3, d3, r3, n3, tmp), r2);
      int n1 = interior(tmp, segment_roots(d1, 4, d2, r2, n2, tmp), r1);
      const int n0 = segment_roots(e, 5, d1, r1, n1, r0);
      const double scale = fabs(e[0]) + fabs(e[1]) + fabs(e[2]) + fabs(e[3]) + fabs(e[5]);
      const double tol = 1e-10 * scale;
      for (int k = 0; k < n1; ++k)
        if (fabs(peval(e, 5, r1[k])) <= tol) amb = 1;
      if (fabs(peval(e, 5, 1.0)) <= tol || fabs(peval(e, 5, -1.0)) <= tol) amb = 1;
      if (scale > 1e8 * fabs(e[5])) amb = 1;
      // candidates: real roots in [-1, 1], then 0, then 1
      double cand[8], rc[8];
      int nc = 0;
      for (int k = 0; k < n0; ++k)
        if (fabs(r0[k]) <= 1.0) cand[nc++] = acos(r0[k]) / M_PI;
      cand[nc++] = 0.0;
      cand[nc++] = 1.0;
      int best = 0;
      for (int k = 0; k < nc; ++k) {
        rc[k] = fit_residual(x, c, cand[k]);
        if (rc[k] < rc[best]) best = k;
      }
      double rs = 0.0;
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const double m = fabs(x[j] - c.b[j]) + fabs(c.a[j]);
        rs += m * m;
      }
      for (int k = 0; k < nc; ++k)
        if (k != best && fabs(cand[k] - cand[best]) > 1e-12 && rc[k] - rc[best] <= 1e-12 * rs)
          amb = 1;
      t_best = cand[best];
    }
    tau[i] = t_best;
    flag[i] = amb;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      // tau . (pi j), the operand order of fit_1D_open_manifold_3D.py:85
      const double cj = cos(t_best * (M_PI * (double)(j + 1)));
      acc[j] = cj * cj;
      acc[3 + j] = cj;
      acc[6 + j] = x[j] * cj;
      acc[9 + j] = x[j];
    }
    acc[12] = amb;
  }
#pragma unroll
  for (int k = 0; k < 13; ++k) red[k][threadIdx.x] = acc[k];
  __syncthreads();
  for (int w = FIT_BLOCK / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w)
#pragma unroll
      for (int k = 0; k < 13; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x < 13) part[blockIdx.x * 13 + threadIdx.x] = red[threadIdx.x][0];
}

// sums[k] = sum over blocks of part[b][k], in block order
__global__ void k_fit1d_sums(const double* __restrict__ part, int nb, double* __restrict__ sums) {
  const int k = threadIdx.x;
  if (k >= 13) return;
  double s = 0.0;
  for (int b = 0; b < nb; ++b) s += part[b * 13 + k];
  sums[k] = s;
}

__global__ void k_zero_d(double* p, int64_t n) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n;
       e += (int64_t)gridDim.x * blockDim.x)
    p[e] = 0.0;
}

}  // namespace memi

using namespace memi;

extern "C" {

int memi_nlsa_condist(const void* D, int d_is_f64, const int64_t* ord, int n, int con_order,
                      double* ConD, void* stream) {
  MEMI_CHECK_ARG(D && ord && ConD, "memi_nlsa_condist: null pointer");
  MEMI_CHECK_ARG(con_order >= 1 && con_order <= CMAX && n > con_order,
                 "memi_nlsa_condist: need 1 <= ConOrder <= %d and n > ConOrder (n=%d, C=%d)",
                 CMAX, n, con_order);
  const int m = n - con_order;
  const int S = CT + con_order - 1;
  const size_t shm = (size_t)S * S * sizeof(double);
  dim3 g((m + CT - 1) / CT, (m + CT - 1) / CT);
  if (d_is_f64)
    hipLaunchKernelGGL(k_condist<double>, g, dim3(256), shm, (hipStream_t)stream,
                       (const double*)D, ord, n, con_order, ConD);
  else
    hipLaunchKernelGGL(k_condist<float>, g, dim3(256), shm, (hipStream_t)stream,
                       (const float*)D, ord, n, con_order, ConD);
  MEMI_CHECK_LAUNCH("k_condist");
  return MEMI_OK;
}

int memi_nlsa_supervectors(const void* spec, const float* ctf_half, int n, int N, int con_order,
                           const double* mu_psi, int ell, double snr, void* out, void* stream) {
  MEMI_CHECK_ARG(spec && ctf_half && mu_psi && out, "memi_nlsa_supervectors: null pointer");
  MEMI_CHECK_ARG(ell >= 1 && ell <= ELLMAX, "memi_nlsa_supervectors: ell=%d must be 1..%d", ell,
                 ELLMAX);
  MEMI_CHECK_ARG(con_order >= 1 && n > con_order && snr > 0,
                 "memi_nlsa_supervectors: bad n=%d ConOrder=%d", n, con_order);
  const int64_t Kh = (int64_t)N * (N / 2 + 1);
  // Delays per wave (9 to 13), and pieces of the steps per wave.  A CU runs eight waves; a step
  // of a workgroup takes its waves per SIMD times 8 sg sums and ~25 other instructions, and each
  // piece starts with its own window sum (C loads) and history.
  const int halves = (ell + 3) / 4;
  const int m = n - con_order;
  int sg = 0, gy = 0, gpb = 0, kshift = 6;
  double best = 0.0;
  for (int g = 13; g >= 9; --g) {
    const int groups = (con_order + g - 1) / g;
    const int y = (groups * halves + 7) / 8;
    const int per = (groups + y - 1) / y;          // delay groups per workgroup: <= 8 waves
    const int64_t res = 256 * (8 / (per * halves));
    for (int ks = 6; ks >= 2; --ks) {
      const int64_t blocks = ((Kh + (1 << ks) - 1) >> ks) * y;
      const double cost = (double)((blocks + res - 1) / res) * (8 / (per * halves)) *
                          ((per * halves + 3) / 4) * (8 * g + 25) *
                          ((double)m / (64 >> ks) + 0.5 * con_order + 2 * g);
      if (sg == 0 || cost < best) {
        best = cost;
        sg = g;
        gy = y;
        gpb = per;
        kshift = ks;
      }
    }
  }
  const int pieces = 64 >> kshift;
  const int steps = (m + pieces - 1) / pieces;
  const int64_t gx = (Kh + (1 << kshift) - 1) >> kshift;
  MEMI_CHECK_ARG(gx < 0x7fffffffLL && gy < 65536, "memi_nlsa_supervectors: too large");
  const dim3 grid((unsigned)gx, (unsigned)gy), block(64 * gpb * halves);
  const bool small = (int64_t)n * Kh < (1LL << 29);      // byte offsets within 32 bits
#define MEMI_SUPERVECTORS(G)                                                                    \
  do {                                                                                          \
    auto kern = small ? k_supervectors<G, uint32_t> : k_supervectors<G, int64_t>;               \
    hipLaunchKernelGGL(kern, grid, block, 0, (hipStream_t)stream, (const float2*)spec, ctf_half, \
                       n, Kh, con_order, mu_psi, ell, snr, kshift, steps, gpb, halves,          \
                       (float2*)out);                                                           \
  } while (0)
  switch (sg) {
    case 9: MEMI_SUPERVECTORS(9); break;
    case 10: MEMI_SUPERVECTORS(10); break;
    case 11: MEMI_SUPERVECTORS(11); break;
    case 12: MEMI_SUPERVECTORS(12); break;
    default: MEMI_SUPERVECTORS(13); break;
  }
#undef MEMI_SUPERVECTORS
  MEMI_CHECK_LAUNCH("k_supervectors");
  return MEMI_OK;
}

int memi_tall_gram(const double* A, int64_t M, int c, double* G, void* stream) {
  MEMI_CHECK_ARG(A && G && M > 0 && c >= 1 && c <= TGMAX, "memi_tall_gram: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_zero_d, dim3(1), dim3(64), 0, s, G, (int64_t)c * c);
  MEMI_CHECK_LAUNCH("k_zero_d");
  hipLaunchKernelGGL(k_tall_gram, dim3(grid_for(M, 256, 2048)), dim3(256), 0, s, A, M, c, G);
  MEMI_CHECK_LAUNCH("k_tall_gram");
  return MEMI_OK;
}

int memi_tall_apply(const double* A, int64_t M, int c, const double* B_host, int d, double* Y,
                    void* stream) {
  MEMI_CHECK_ARG(A && B_host && Y && M > 0 && c >= 1 && c <= TGMAX && d >= 1 && d <= TGMAX,
                 "memi_tall_apply: bad arguments");
  SmallMat B{};
  for (int e = 0; e < c * d; ++e) B.v[e] = B_host[e];
  hipLaunchKernelGGL(k_tall_apply, dim3(grid_for(M)), dim3(256), 0, (hipStream_t)stream, A, M, c,
                     B, d, Y);
  MEMI_CHECK_LAUNCH("k_tall_apply");
  return MEMI_OK;
}

int memi_center_gram(double* U2, int64_t npix, int q_dim, double* G, void* stream) {
  MEMI_CHECK_ARG(U2 && G && npix > 0 && q_dim >= 1 && q_dim <= 4096,
                 "memi_center_gram: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  // column sums are accumulated in G's first q_dim entries before G is cleared for the Gram
  hipLaunchKernelGGL(k_zero_d, dim3(grid_for((int64_t)q_dim * q_dim)), dim3(256), 0, s, G,
                     (int64_t)q_dim * q_dim);
  MEMI_CHECK_LAUNCH("k_zero_d");
  dim3 gs(256, (unsigned)((q_dim + 255) / 256));
  hipLaunchKernelGGL(k_col_sum, gs, dim3(256), 0, s, U2, npix, q_dim, G);
  MEMI_CHECK_LAUNCH("k_col_sum");
  hipLaunchKernelGGL(k_col_center, dim3(grid_for(npix * q_dim)), dim3(256), 0, s, U2, npix,
                     q_dim, G);
  MEMI_CHECK_LAUNCH("k_col_center");
  hipLaunchKernelGGL(k_zero_d, dim3(1), dim3(256), 0, s, G, (int64_t)q_dim);
  MEMI_CHECK_LAUNCH("k_zero_d");
  dim3 gg((unsigned)((q_dim + 15) / 16), (unsigned)((q_dim + 15) / 16),
          (unsigned)((npix + 4 * GC_ROWS - 1) / (4 * GC_ROWS)));
  hipLaunchKernelGGL(k_gram_cols, gg, dim3(256), 0, s, U2, npix, q_dim, G);
  MEMI_CHECK_LAUNCH("k_gram_cols");
  return MEMI_OK;
}

int memi_nlsa_imgt(const double* Ubar, const double* H, const double* inv_sd, int64_t npix,
                   int q_dim, int ncols, double* IMGT, void* stream) {
  MEMI_CHECK_ARG(Ubar && H && inv_sd && IMGT && npix > 0 && q_dim > 0 && ncols > 0,
                 "memi_nlsa_imgt: bad arguments");
  dim3 g((unsigned)((ncols + IM_J - 1) / IM_J), (unsigned)((npix + IM_P - 1) / IM_P));
  hipLaunchKernelGGL(k_imgt, g, dim3(256), 0, (hipStream_t)stream, Ubar, H, inv_sd, npix, q_dim,
                     ncols, IMGT);
  MEMI_CHECK_LAUNCH("k_imgt");
  return MEMI_OK;
}

int memi_nlsa_recon_dist(const double* Gq, const double* H, int q_dim, int ncols, int64_t npix,
                         double* inv_sd, float* Drecon2, double* ws, void* stream) {
  MEMI_CHECK_ARG(Gq && H && inv_sd && Drecon2 && ws && q_dim > 0 && q_dim <= 4096 &&
                     ncols > 0 && npix > 0,
                 "memi_nlsa_recon_dist: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  double* T = ws;
  double* dg = ws + (int64_t)q_dim * ncols;
  hipLaunchKernelGGL(k_gq_h, dim3((ncols + 255) / 256, q_dim), dim3(256), 0, s, Gq, H, q_dim,
                     ncols, T);
  MEMI_CHECK_LAUNCH("k_gq_h");
  hipLaunchKernelGGL(k_recon_diag, dim3((ncols + 255) / 256), dim3(256), 0, s, H, T, q_dim, ncols,
                     (double)npix, dg, inv_sd);
  MEMI_CHECK_LAUNCH("k_recon_diag");
  const unsigned nt = (unsigned)((ncols + 63) / 64);
  hipLaunchKernelGGL(k_recon_dist, dim3(nt, nt), dim3(256), 0, s, H, T, dg, inv_sd, q_dim, ncols,
                     Drecon2);
  MEMI_CHECK_LAUNCH("k_recon_dist");
  return MEMI_OK;
}

int memi_fit1d_tau(const double* x, int n, const double* ab_host, double* tau, int32_t* flag,
                   double* sums, double* ws, void* stream) {
  MEMI_CHECK_ARG(x && ab_host && tau && flag && sums && ws && n > 0,
                 "memi_fit1d_tau: bad arguments");
  FitCurve c;
  for (int j = 0; j < 3; ++j) {
    c.a[j] = ab_host[j];
    c.b[j] = ab_host[3 + j];
  }
  const int nb = (n + FIT_BLOCK - 1) / FIT_BLOCK;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_fit1d_tau, dim3(nb), dim3(FIT_BLOCK), 0, s, x, n, c, tau, flag, ws);
  MEMI_CHECK_LAUNCH("k_fit1d_tau");
  hipLaunchKernelGGL(k_fit1d_sums, dim3(1), dim3(64), 0, s, ws, nb, sums);
  MEMI_CHECK_LAUNCH("k_fit1d_sums");
  return MEMI_OK;
}

}  // extern "C"
