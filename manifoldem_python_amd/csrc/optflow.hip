// Optical flow of NLSA movies (the CC stage): 3-D Perona-Malik diffusion of each movie, block
// averaging of its frames, Gaussian low-pass, Horn-Schunck flow between consecutive averaged
// frames, and the sum of the flows with its orientation and magnitude.
//
// Reference: CC/hornschunck_simple.py:9-84, CC/OpticalFlowMovie.py:21-24, 202-341, 385-555.
//
// The kernels reproduce the reference's arithmetic: float32 where numpy computes in float32
// (the diffusion, the derivative images, the denominator alpha^2 + fx^2 + fy^2), float64
// accumulation rounded once to the output type where scipy.ndimage filters (it accumulates each
// output in double), and the reference's operation order with floating-point contraction off.
// Two take another order: the float64 Horn-Schunck iterations (k_hs_strips: a separable average by
// fma and no division; within 1e-13 of the flow's scale after 200 iterations) and the quotients by
// constants in the diffusion (products with float64 reciprocals, the same float32 values).
// Boundaries are scipy's mode 'reflect' (half-sample mirror), which at distance 1 is a clamp.
//
// Data layout: a batch of movies is (movie, frame, row, column) row-major; each frame is the
// reference's Mov[f] = np.resize(row, (dim, dim)).
#include "common.h"

namespace memi {

// --- 3-D anisotropic diffusion (OpticalFlowMovie.py:270-336) -----------------------------------

// g(delta) * delta of one face: option 1 exp(-(d/kappa)^2)/step, option 2 1/(1+(d/kappa)^2)/step.
// numpy evaluates the float32 exp; here it is the float64 exp rounded to float32.  The quotients
// by the constants kappa and step are products with their float64 reciprocals, rounded once: a
// quotient of two float32 numbers is never nearer than 2^-49 (relative) to a rounding boundary
// of float32, and the product is within 2^-52 of it, so these are the float32 quotients.  (A
// subnormal quotient may differ in its last bit; d/kappa is squared and a flux of that size
// changes no voxel.)
template <int OPTION>
__device__ inline float pm_flux(float d, double rkappa, double rstep) {
#pragma clang fp contract(off)
  const float q = (float)((double)d * rkappa);
  const float q2 = q * q;
  float g;
  if (OPTION == 1) g = (float)exp(-(double)q2);
  else g = 1.0f / (1.0f + q2);
  g = (float)((double)g * rstep);
  return g * d;
}

// One update of every voxel: out = s + gamma * ((UD + NS) + EW), where UD = D(z) - D(z-1) with
// D(z) = g(s[z+1]-s[z]) (s[z+1]-s[z]) for z < F-1 and 0 on the last frame (no flux through the
// stack's faces); NS along rows, EW along columns alike.
//
// Bound: the float64 exp of every face (8 B of traffic per voxel take 85 us at 52 M voxels).  Each
// face's flux is computed once: a thread walks its pixel through zc frames and keeps the flux
// behind it, and the fluxes above and to the left come through LDS from the thread that owns
// them, except for a block's first row of pixels.  52 M voxels: 0.28 ms per step, 0.51 ms with
// both faces' fluxes computed by every voxel and two float32 divisions per flux.
constexpr int kAnisoThreads = 1024;

template <int OPTION>
__global__ __launch_bounds__(kAnisoThreads) void k_anisodiff_step(
    const float* __restrict__ in, float* __restrict__ out, int F, int H, int W, int nblk, int nz,
    int zc, double rkappa, float gamma, double rs0, double rs1, double rs2) {
#pragma clang fp contract(off)
  __shared__ float fl[2][2][kAnisoThreads];
  const int tid = threadIdx.x;
  const int64_t plane = (int64_t)H * W;
  const int64_t m = blockIdx.x / ((unsigned)nblk * nz);
  const int r = (int)(blockIdx.x % ((unsigned)nblk * nz));
  const int64_t p = (int64_t)(r % nblk) * kAnisoThreads + tid;
  const int z0 = (r / nblk) * zc, z1 = min(z0 + zc, F);
  const int64_t pp = min(p, plane - 1);      // threads past the plane repeat its last pixel
  const int x = (int)(pp % W), y = (int)(pp / W);
  const int64_t base = (m * F + z0) * plane + pp;
  const float* src = in + base;
  float* dst = out + base;
  float c = src[0];
  float Dp = z0 > 0 ? pm_flux<OPTION>(c - src[-plane], rkappa, rs0) : 0.0f;
  for (int z = z0; z < z1; ++z) {
    float(*f)[kAnisoThreads] = fl[z & 1];
    const float next = z < F - 1 ? src[plane] : c;
    const float Sy = y < H - 1 ? pm_flux<OPTION>(src[W] - c, rkappa, rs1) : 0.0f;
    const float Ex = x < W - 1 ? pm_flux<OPTION>(src[1] - c, rkappa, rs2) : 0.0f;
    f[0][tid] = Sy;
    f[1][tid] = Ex;
    const float Dz = z < F - 1 ? pm_flux<OPTION>(next - c, rkappa, rs0) : 0.0f;
    __syncthreads();
    const float UD = z > 0 ? Dz - Dp : Dz;
    float NS = Sy, EW = Ex;
    if (y > 0) NS = Sy - (tid >= W ? f[0][tid - W] : pm_flux<OPTION>(c - src[-W], rkappa, rs1));
    if (x > 0) EW = Ex - (tid >= 1 ? f[1][tid - 1] : pm_flux<OPTION>(c - src[-1], rkappa, rs2));
    if (p < plane) *dst = c + gamma * ((UD + NS) + EW);
    Dp = Dz;
    c = next;
    src += plane;
    dst += plane;
  }
}

// --- block averages of frames (OpticalFlowMovie.py:447-457) -------------------------------------

// out[m][b][p] = (sum of in[m][f][p] over the block's frames, in frame order, float64) / count:
// the float64 np.mean of float32 frames.
__global__ void k_block_average(const float* __restrict__ in, int64_t nmov, int F, int64_t hw,
                                int bs, int A, double* __restrict__ out) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= nmov * A * hw) return;
  const int64_t p = t % hw;
  const int64_t mb = t / hw;
  const int b = (int)(mb % A);
  const int64_t m = mb / A;
  const int f0 = b * bs;
  const int f1 = min(f0 + bs, F);
  const float* src = in + (m * F + f0) * hw + p;
  double s = (double)src[0];
  for (int f = 1; f < f1 - f0; ++f) s += (double)src[(int64_t)f * hw];
  out[t] = s / (double)(f1 - f0);
}

// --- Gaussian low-pass (hornschunck_simple.py:35-38, scipy gaussian_filter) ---------------------

constexpr int kGaussMaxR = 32;
struct GaussTaps {
  double w[kGaussMaxR + 1];  // w[d] = weight at distance d (normalised, symmetric)
  int r;
};

__device__ inline int reflect_index(int i, int n) {
  const int m = 2 * n;
  i %= m;
  if (i < 0) i += m;
  return i < n ? i : m - 1 - i;
}

// One separable pass along AXIS (0: down the rows, 1: along a row).  The input is first rounded
// to the output type (the reference casts before it filters; the second pass reads the first's
// output), then out = w0 c + sum_{d = r..1} (in[-d] + in[+d]) w_d in float64, rounded once.
template <typename TI, typename TO, int AXIS>
__global__ void k_gauss_pass(const TI* __restrict__ in, TO* __restrict__ out, int64_t count,
                             int H, int W, GaussTaps g) {
#pragma clang fp contract(off)
  const int64_t hw = (int64_t)H * W;
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= count * hw) return;
  const int x = (int)(t % W);
  const int y = (int)((t / W) % H);
  const TI* img = in + (t / hw) * hw;
  auto ld = [&](int yy, int xx) { return (double)(TO)img[(int64_t)yy * W + xx]; };
  double acc = ld(y, x) * g.w[0];
  for (int d = g.r; d >= 1; --d) {
    double a, b;
    if (AXIS == 0) {
      a = ld(reflect_index(y - d, H), x);
      b = ld(reflect_index(y + d, H), x);
    } else {
      a = ld(y, reflect_index(x - d, W));
      b = ld(y, reflect_index(x + d, W));
    }
    acc += (a + b) * g.w[d];
  }
  out[t] = (TO)acc;
}

// --- Horn-Schunck derivatives (hornschunck_simple.py:24-31) ------------------------------------

// scipy's convolve with a 2 x 2 kernel k: out[i][j] = k11 a[i][j] + k10 a[i][j+1]
// + k01 a[i+1][j] + k00 a[i+1][j+1] (float64, rounded to float32), the last row and column
// mirrored onto themselves.  fx, fy, ft are float32 sums of the two frames' convolutions.
__global__ void k_hs_derivatives(const float* __restrict__ frames,
                                 const int32_t* __restrict__ pairs, int64_t nP, int H, int W,
                                 float* __restrict__ fx, float* __restrict__ fy,
                                 float* __restrict__ ft) {
#pragma clang fp contract(off)
  const int64_t hw = (int64_t)H * W;
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= nP * hw) return;
  const int x = (int)(t % W);
  const int y = (int)((t / W) % H);
  const int64_t p = t / hw;
  const int x1 = min(x + 1, W - 1);
  const int y1 = min(y + 1, H - 1);
  double v[2][4];
  for (int f = 0; f < 2; ++f) {
    const float* im = frames + (int64_t)pairs[2 * p + f] * hw;
    v[f][0] = im[(int64_t)y * W + x];
    v[f][1] = im[(int64_t)y * W + x1];
    v[f][2] = im[(int64_t)y1 * W + x];
    v[f][3] = im[(int64_t)y1 * W + x1];
  }
  float cx[2], cy[2], ct[2];
  for (int f = 0; f < 2; ++f) {
    double s = 0.0;
    s += 0.25 * v[f][0]; s += -0.25 * v[f][1]; s += 0.25 * v[f][2]; s += -0.25 * v[f][3];
    cx[f] = (float)s;
    s = 0.0;
    s += 0.25 * v[f][0]; s += 0.25 * v[f][1]; s += -0.25 * v[f][2]; s += -0.25 * v[f][3];
    cy[f] = (float)s;
    const double kt = f == 0 ? 0.25 : -0.25;
    s = 0.0;
    s += kt * v[f][0]; s += kt * v[f][1]; s += kt * v[f][2]; s += kt * v[f][3];
    ct[f] = (float)s;
  }
  fx[t] = cx[0] + cx[1];
  fy[t] = cy[0] + cy[1];
  ft[t] = ct[0] + ct[1];
}

// --- Horn-Schunck iterations (hornschunck_simple.py:70-82) -------------------------------------

// `iters` (<= R) iterations per launch on a TS x TS output tile, temporally blocked in LDS: the
// tile plus an R-pixel halo of U, V, fx, fy, ft is loaded once; sub-iteration s updates the
// cells within iters - s of the tile (their 3 x 3 neighbours were updated by sub-iteration
// s - 1), so after `iters` sub-iterations the tile holds the exact iterate.  A neighbour outside
// the image is the nearest edge cell (mode 'reflect' at distance 1).  Used for float32 flows,
// which round uAvg and every later operation to float32; float64 flows run on k_hs_strips.
//
//   uAvg = sum of the 8 neighbours x HSKERN (scipy's raster order, float64, rounded to float32)
//   der  = ((fx uAvg + fy vAvg) + ft) / den,   den = (float)((alpha^2 + fx^2) + fy^2)
//   U = uAvg - fx der,  V = vAvg - fy der       (in float32, as numpy promotes a float32 start)
template <int TS, int R, int NT>
__global__ __launch_bounds__(NT) void k_hs_iterate(
    const float* __restrict__ gfx, const float* __restrict__ gfy, const float* __restrict__ gft,
    int H, int W, int tiles_x, int ntiles, float alpha2, int iters,
    const float* __restrict__ Uin, const float* __restrict__ Vin, float* __restrict__ Uout,
    float* __restrict__ Vout) {
#pragma clang fp contract(off)
  constexpr int E = TS + 2 * R;
  constexpr int NC = E * E;
  constexpr int PER = (NC + NT - 1) / NT;
  __shared__ float sU[NC];
  __shared__ float sV[NC];
  __shared__ float sfx[NC];
  __shared__ float sfy[NC];
  __shared__ float sft[NC];
  const int64_t p = blockIdx.x / ntiles;
  const int tile = (int)(blockIdx.x % ntiles);
  const int ty0 = (tile / tiles_x) * TS;
  const int tx0 = (tile % tiles_x) * TS;
  const int64_t base = p * (int64_t)H * W;

  // per owned cell: LDS index, image coordinates, Chebyshev distance to the tile (-1: outside
  // the image)
  int dist[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = threadIdx.x + k * NT;
    const int ly = c / E, lx = c % E;
    const int gy = ty0 - R + ly, gx = tx0 - R + lx;
    int d = -1;
    if (c < NC && gy >= 0 && gy < H && gx >= 0 && gx < W) {
      const int dy = max(max(ty0 - gy, gy - (ty0 + TS - 1)), 0);
      const int dx = max(max(tx0 - gx, gx - (tx0 + TS - 1)), 0);
      d = max(dy, dx);
    }
    dist[k] = d;
    if (d >= 0 && d <= iters) {
      const int64_t g = base + (int64_t)gy * W + gx;
      sU[c] = Uin[g];
      sV[c] = Vin[g];
      sfx[c] = gfx[g];
      sfy[c] = gfy[g];
      sft[c] = gft[g];
    }
  }
  __syncthreads();

  constexpr double w1 = 1.0 / 12, w2 = 1.0 / 6;
  for (int s = 1; s <= iters; ++s) {
    float nu[PER], nv[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int c = threadIdx.x + k * NT;
      if (dist[k] >= 0 && dist[k] <= iters - s) {
        const int ly = c / E, lx = c % E;
        const int gy = ty0 - R + ly, gx = tx0 - R + lx;
        const int up = gy > 0 ? -E : 0, dn = gy < H - 1 ? E : 0;
        const int lf = gx > 0 ? -1 : 0, rt = gx < W - 1 ? 1 : 0;
        double au = 0.0, av = 0.0;
        au += (double)sU[c + up + lf] * w1; av += (double)sV[c + up + lf] * w1;
        au += (double)sU[c + up] * w2;      av += (double)sV[c + up] * w2;
        au += (double)sU[c + up + rt] * w1; av += (double)sV[c + up + rt] * w1;
        au += (double)sU[c + lf] * w2;      av += (double)sV[c + lf] * w2;
        au += (double)sU[c + rt] * w2;      av += (double)sV[c + rt] * w2;
        au += (double)sU[c + dn + lf] * w1; av += (double)sV[c + dn + lf] * w1;
        au += (double)sU[c + dn] * w2;      av += (double)sV[c + dn] * w2;
        au += (double)sU[c + dn + rt] * w1; av += (double)sV[c + dn + rt] * w1;
        const float ua = (float)au, va = (float)av;
        const float fx = sfx[c], fy = sfy[c];
        const float den = (alpha2 + fx * fx) + fy * fy;
        const float der = ((fx * ua + fy * va) + sft[c]) / den;
        nu[k] = ua - fx * der;
        nv[k] = va - fy * der;
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int c = threadIdx.x + k * NT;
      if (dist[k] >= 0 && dist[k] <= iters - s) {
        sU[c] = nu[k];
        sV[c] = nv[k];
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    if (dist[k] == 0) {
      const int c = threadIdx.x + k * NT;
      const int gy = ty0 - R + c / E, gx = tx0 - R + c % E;
      const int64_t g = base + (int64_t)gy * W + gx;
      Uout[g] = sU[c];
      Vout[g] = sV[c];
    }
  }
}

// Float64 iterations on register strips.  A wave owns S rows x 64 C columns of one frame pair
// (each lane C neighbouring columns) and keeps U, V and the scaled derivatives
//   (gx, gy, gt) = (fx, fy, ft) / sqrt(den)
// in registers for `iters` iterations, so that
//   U = uAvg - gx d,  V = vAvg - gy d,  d = (gx uAvg + gy vAvg) + gt
// needs no division.  HSKERN separates: with p(x) = w2 c + w1 a, a = up + down and c the cell
// itself, uAvg = w2 a(x) + p(x - 1) + p(x + 1), so one value per cell crosses to each side: by a
// register move between a lane's own columns, by a DPP wave shift at the lane's edge.  Rows
// cross between waves through LDS, two per wave and iteration (double buffered, one barrier).
// NW waves stack to a band of NW S rows.  A band that does not hold the whole image keeps a halo
// of `iters` rows (and columns) on each open side, whose cells go stale one per iteration.
//
// Bound: neither the vector units nor memory alone.  At 128 x 128 the SIMDs issue vector
// instructions on 56 % of their cycles (64 % of those in float64, the rest register moves), and a
// launch moves 0.39 GB of U, V, fx, fy, ft, a quarter of its 0.30 ms at a large copy's rate; the
// 128 KB of LDS leave one workgroup per CU, so nothing runs beside a tile's loads, stores and
// barriers.  Eight cells per lane at 10 registers each leave four waves per SIMD: 640 pairs of
// 128 x 128, 200 iterations take 3.85 ms in 13 launches of three tiles per pair (16 cells and two
// waves per SIMD: 3.96; the LDS-tile form above, which reads 16 float64 neighbours per cell from LDS
// and divides: 11.6).
// Two columns per lane halve the DPP moves (one column: 4.08 ms), one suits narrow images; three
// (5 rows, 40-row bands) were slower at 128 columns (6.9 ms) and at 160 (9.2 against 8.7).
constexpr int kHsWaves = 16;
constexpr int hs_strip_rows(int cols) { return 8 / cols; }

// nx x ny tiles of an image.  Along a side with several tiles, tile i loads from cell i ow on; it
// writes from halo cells further on (the first tile from the image's edge) up to the next tile's
// first written cell (the last tile up to the image's edge).  With one tile ow is unused.  halo: iterations per launch (0: one tile holds the image).
struct HsTiling {
  int nx, ny;
  int ow, oh;
  int halo;
};

template <int C, int S>
__global__ __launch_bounds__(kHsWaves * 64) void k_hs_strips(
    const float* __restrict__ gfx, const float* __restrict__ gfy, const float* __restrict__ gft,
    int H, int W, HsTiling t, float alpha2, int iters, const double* Uin, const double* Vin,
    double* Uout, double* Vout) {
#pragma clang fp contract(off)
  constexpr int NW = kHsWaves, LW = 64 * C;
  __shared__ double rows[2][NW][2][2][LW];   // parity, wave, top / bottom row, U / V, column
  const int tile = (int)(blockIdx.x % (unsigned)(t.nx * t.ny));
  const int64_t base = (int64_t)(blockIdx.x / (unsigned)(t.nx * t.ny)) * H * W;
  const int tx = tile % t.nx, ty = tile / t.nx;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int x0 = tx * t.ow + lane * C, yw = ty * t.oh + w * S;
  double U[S][C], V[S][C], gx[S][C], gy[S][C], gt[S][C];
#pragma unroll
  for (int s = 0; s < S; ++s) {
#pragma unroll
    for (int j = 0; j < C; ++j) {
      // cells outside the image are loaded as its edge cells; they reach no cell inside
      const int64_t g = base + (int64_t)min(yw + s, H - 1) * W + min(x0 + j, W - 1);
      U[s][j] = Uin[g];
      V[s][j] = Vin[g];
      const float fx = gfx[g], fy = gfy[g], ft = gft[g];
      const float den = (alpha2 + fx * fx) + fy * fy;
      const double r = rsqrt((double)den);
      gx[s][j] = fx * r;
      gy[s][j] = fy * r;
      gt[s][j] = ft * r;
    }
  }
  // Columns beyond the image pass zero to their neighbours (their weights are zero), the wave's
  // outer lanes read zero past its ends, and a column at the image's edge adds its own p (edge)
  // for the neighbour it lacks.
  double w1[C], w2[C], edge[C];
#pragma unroll
  for (int j = 0; j < C; ++j) {
    w1[j] = x0 + j < W ? 1.0 / 12 : 0.0;
    w2[j] = x0 + j < W ? 1.0 / 6 : 0.0;
    edge[j] = (x0 + j == 0 ? 1.0 : 0.0) + (x0 + j == W - 1 ? 1.0 : 0.0);
  }
  const int s_last = H - 1 - yw;             // the image's last row within the strip
  // row s from the rows above and below it
  auto update = [&](int s, const double* up_u, const double* up_v, const double* dn_u,
                    const double* dn_v) {
    double au[C], av[C], qu[C], qv[C];
#pragma unroll
    for (int j = 0; j < C; ++j) {
      au[j] = up_u[j] + dn_u[j];
      av[j] = up_v[j] + dn_v[j];
      qu[j] = fma(w1[j], au[j], w2[j] * U[s][j]);
      qv[j] = fma(w1[j], av[j], w2[j] * V[s][j]);
    }
    const double lu = dpp_move<0x138, 0xf>(qu[C - 1]);             // wave_shr:1
    const double lv = dpp_move<0x138, 0xf>(qv[C - 1]);
    const double ru = dpp_move<0x130, 0xf>(qu[0]);                 // wave_shl:1
    const double rv = dpp_move<0x130, 0xf>(qv[0]);
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const double l_u = j == 0 ? lu : qu[j > 0 ? j - 1 : 0];
      const double l_v = j == 0 ? lv : qv[j > 0 ? j - 1 : 0];
      const double r_u = j == C - 1 ? ru : qu[j < C - 1 ? j + 1 : j];
      const double r_v = j == C - 1 ? rv : qv[j < C - 1 ? j + 1 : j];
      const double ua = fma(edge[j], qu[j], fma(1.0 / 6, au[j], l_u) + r_u);
      const double va = fma(edge[j], qv[j], fma(1.0 / 6, av[j], l_v) + r_v);
      const double d = fma(gx[s][j], ua, fma(gy[s][j], va, gt[s][j]));
      U[s][j] = fma(-gx[s][j], d, ua);
      V[s][j] = fma(-gy[s][j], d, va);
    }
    __builtin_amdgcn_sched_barrier(0);       // row by row: interleaved rows overflow the registers
  };
  for (int it = 0; it < iters; ++it) {
    double(*rb)[2][2][LW] = rows[it & 1];
#pragma unroll
    for (int j = 0; j < C; ++j) {
      rb[w][0][0][j * 64 + lane] = U[0][j];
      rb[w][0][1][j * 64 + lane] = V[0][j];
      rb[w][1][0][j * 64 + lane] = U[S - 1][j];
      rb[w][1][1][j * 64 + lane] = V[S - 1][j];
    }
    // the row below the image's last one repeats it
#pragma unroll
    for (int s = 0; s + 1 < S; ++s)
      if (s == s_last) {
#pragma unroll
        for (int j = 0; j < C; ++j) {
          U[s + 1][j] = U[s][j];
          V[s + 1][j] = V[s][j];
        }
      }
    __syncthreads();
    double pu[C], pv[C], nu[C], nv[C];       // the row above; the row below the strip
#pragma unroll
    for (int j = 0; j < C; ++j) {
      // the first wave's strip starts at the image's top or in the halo, the last one's ends at
      // its bottom or in the halo
      const bool top = w == 0, bottom = w == NW - 1 || s_last == S - 1;
      pu[j] = top ? U[0][j] : rb[top ? w : w - 1][1][0][j * 64 + lane];
      pv[j] = top ? V[0][j] : rb[top ? w : w - 1][1][1][j * 64 + lane];
      nu[j] = bottom ? U[S - 1][j] : rb[w + 1 < NW ? w + 1 : w][0][0][j * 64 + lane];
      nv[j] = bottom ? V[S - 1][j] : rb[w + 1 < NW ? w + 1 : w][0][1][j * 64 + lane];
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
      double cu[C], cv[C];
#pragma unroll
      for (int j = 0; j < C; ++j) {
        cu[j] = U[s][j];
        cv[j] = V[s][j];
      }
      if (s + 1 < S) update(s, pu, pv, U[s + 1 < S ? s + 1 : s], V[s + 1 < S ? s + 1 : s]);
      else update(s, pu, pv, nu, nv);
#pragma unroll
      for (int j = 0; j < C; ++j) {
        pu[j] = cu[j];
        pv[j] = cv[j];
      }
    }
  }
  const int ox = tx ? tx * t.ow + t.halo : 0, oy = ty ? ty * t.oh + t.halo : 0;
  const int ex = tx == t.nx - 1 ? W : (tx + 1) * t.ow + t.halo;
  const int ey = ty == t.ny - 1 ? H : (ty + 1) * t.oh + t.halo;
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const int x = x0 + j, y = yw + s;
      if (x >= ox && x < ex && y >= oy && y < ey) {
        const int64_t g = base + (int64_t)y * W + x;
        Uout[g] = U[s][j];
        Vout[g] = V[s][j];
      }
    }
}

// Tiles of one side: n tiles of `cap` cells with a halo of R on each open side cover L cells when
// L <= n cap - 2 (n - 1) R (the two end tiles have one open side each).  The largest such R for
// n tiles, at most `niter`.
inline int hs_halo(int L, int cap, int n, int niter) {
  if (n == 1) return L <= cap ? niter : 0;
  const int64_t r = ((int64_t)n * cap - L) / (2 * (n - 1));
  return (int)std::max<int64_t>(0, std::min<int64_t>({r, (cap - 1) / 2, niter}));
}

// --- flow sum, orientation, magnitude (OpticalFlowMovie.py:21-24, 519-555) ----------------------

// numpy's remainder x % 2.0 (result in [0, 2), a zero remainder is +0)
__device__ inline double py_mod2(double a) {
  double m = fmod(a, 2.0);
  if (m != 0.0) {
    if (m < 0.0) m += 2.0;
  } else {
    m = 0.0;
  }
  return m;
}

// VxM = 0 + U[0] + U[1] + ... over a movie's frame pairs (float64, in order; from_zero = 0 starts
// from U[0] itself, keeping a -0.0), orient = (atan2(VyM, VxM) % 2) pi, mag = sqrt(Vx^2 + Vy^2),
// orient_rev = the orientation of (-VxM, -VyM).
template <typename T>
__global__ void k_flow_sum(const T* __restrict__ U, const T* __restrict__ V, int64_t nmov, int A,
                           int64_t hw, int from_zero, double* __restrict__ vx,
                           double* __restrict__ vy, double* __restrict__ orient,
                           double* __restrict__ mag, double* __restrict__ orient_rev) {
#pragma clang fp contract(off)
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= nmov * hw) return;
  const int64_t m = t / hw, p = t % hw;
  double sx, sy;
  int a0;
  if (from_zero) {
    sx = 0.0; sy = 0.0; a0 = 0;
  } else {
    sx = (double)U[m * A * hw + p]; sy = (double)V[m * A * hw + p]; a0 = 1;
  }
  for (int a = a0; a < A; ++a) {
    sx = sx + (double)U[(m * A + a) * hw + p];
    sy = sy + (double)V[(m * A + a) * hw + p];
  }
  vx[t] = sx;
  vy[t] = sy;
  if (orient) orient[t] = py_mod2(atan2(sy, sx)) * M_PI;
  if (mag) mag[t] = sqrt(sx * sx + sy * sy);
  if (orient_rev) orient_rev[t] = py_mod2(atan2(-sy, -sx)) * M_PI;
}

constexpr int kHsTile = 32;
constexpr int kHsHalo = 4;
constexpr int kHsThreads = 256;

}  // namespace memi

using namespace memi;

extern "C" {

int memi_flow_anisodiff(const float* in, float* out, float* tmp, int64_t nmov, int F, int H,
                        int W, int niter, double kappa, double gamma, double step0, double step1,
                        double step2, int option, void* stream) {
  MEMI_CHECK_ARG(in && out, "memi_flow_anisodiff: null pointer");
  MEMI_CHECK_ARG(nmov >= 0 && F >= 1 && H >= 1 && W >= 1,
                 "memi_flow_anisodiff: bad sizes nmov=%lld F=%d H=%d W=%d", (long long)nmov, F,
                 H, W);
  MEMI_CHECK_ARG(option == 1 || option == 2, "memi_flow_anisodiff: option must be 1 or 2");
  MEMI_CHECK_ARG(in != out, "memi_flow_anisodiff: in and out must not alias");
  const int steps = niter - 1;  // the reference's loop runs over range(1, niter)
  MEMI_CHECK_ARG(steps < 2 || (tmp && tmp != in && tmp != out),
                 "memi_flow_anisodiff: tmp buffer needed for niter > 2");
  const int64_t nvox = nmov * F * (int64_t)H * W;
  hipStream_t s = (hipStream_t)stream;
  if (nvox == 0) return MEMI_OK;
  if (steps <= 0) {
    if (hipMemcpyAsync(out, in, nvox * sizeof(float), hipMemcpyDeviceToDevice, s) != hipSuccess) {
      set_error("memi_flow_anisodiff: copy failed");
      return MEMI_ELAUNCH;
    }
    return MEMI_OK;
  }
  // the last step writes `out`
  float* buf[2];
  buf[(steps - 1) % 2] = out;
  buf[steps % 2] = tmp;
  // frames per thread: all of them when the batch alone gives every CU its two blocks twice over,
  // else fewer (each further piece computes one more face per pixel)
  const int64_t nblk = ((int64_t)H * W + kAnisoThreads - 1) / kAnisoThreads;
  const int64_t want = std::min<int64_t>(F, std::max<int64_t>(1, 1024 / (nmov * nblk)));
  const int zc = (int)((F + want - 1) / want);
  const int nz = (F + zc - 1) / zc;
  MEMI_CHECK_ARG(nblk * nz <= 0x7fffffffLL / nmov, "memi_flow_anisodiff: batch too large");
  const dim3 grid((unsigned)(nmov * nblk * nz));
  const float k32 = (float)kappa, s0 = (float)step0, s1 = (float)step1, s2 = (float)step2;
  const double rk = 1.0 / k32, r0 = 1.0 / s0, r1 = 1.0 / s1, r2 = 1.0 / s2;
  for (int k = 0; k < steps; ++k) {
    const float* src = k == 0 ? in : buf[(k - 1) % 2];
    float* dst = buf[k % 2];
    if (option == 1)
      hipLaunchKernelGGL(k_anisodiff_step<1>, grid, dim3(kAnisoThreads), 0, s, src, dst, F, H, W,
                         (int)nblk, nz, zc, rk, (float)gamma, r0, r1, r2);
    else
      hipLaunchKernelGGL(k_anisodiff_step<2>, grid, dim3(kAnisoThreads), 0, s, src, dst, F, H, W,
                         (int)nblk, nz, zc, rk, (float)gamma, r0, r1, r2);
    MEMI_CHECK_LAUNCH("k_anisodiff_step");
  }
  return MEMI_OK;
}

int memi_flow_block_average(const float* in, int64_t nmov, int F, int64_t hw, int bs,
                            double* out, void* stream) {
  MEMI_CHECK_ARG(in && out, "memi_flow_block_average: null pointer");
  MEMI_CHECK_ARG(nmov >= 0 && F >= 1 && hw >= 1 && bs >= 1,
                 "memi_flow_block_average: bad sizes nmov=%lld F=%d hw=%lld bs=%d",
                 (long long)nmov, F, (long long)hw, bs);
  const int A = (F + bs - 1) / bs;
  const int64_t n = nmov * A * hw;
  if (n == 0) return MEMI_OK;
  hipLaunchKernelGGL(k_block_average, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, in, nmov, F, hw, bs, A, out);
  MEMI_CHECK_LAUNCH("k_block_average");
  return MEMI_OK;
}

int memi_gaussian_filter(const void* in, int in_f64, void* out, int out_f64, void* tmp,
                         int64_t count, int H, int W, double sigma, void* stream) {
  MEMI_CHECK_ARG(in && out && tmp, "memi_gaussian_filter: null pointer");
  MEMI_CHECK_ARG(count >= 0 && H >= 1 && W >= 1, "memi_gaussian_filter: bad sizes");
  MEMI_CHECK_ARG(in_f64 || !out_f64,
                 "memi_gaussian_filter: float32 input with float64 output is not a reference "
                 "case");
  MEMI_CHECK_ARG(tmp != in && tmp != out, "memi_gaussian_filter: tmp must not alias");
  MEMI_CHECK_ARG(sigma > 0.0, "memi_gaussian_filter: sigma must be positive");
  // scipy: radius = int(truncate * sigma + 0.5) with truncate 4, weights exp(-x^2 / (2 sigma^2))
  // normalised to sum 1
  const int r = (int)(4.0 * sigma + 0.5);
  MEMI_CHECK_ARG(r <= kGaussMaxR, "memi_gaussian_filter: sigma %.3f needs radius %d > %d", sigma,
                 r, kGaussMaxR);
  GaussTaps g{};
  g.r = r;
  double raw[2 * kGaussMaxR + 1];
  const int n_taps = 2 * r + 1;
  const double c = -0.5 / (sigma * sigma);
  for (int i = -r; i <= r; ++i) raw[i + r] = std::exp(c * (double)(i * i));
  // numpy's sum of up to 128 values: a plain loop below 8, else 8 strided partial sums combined
  // pairwise, then the tail
  double sum = 0.0;
  if (n_taps < 8) {
    for (int i = 0; i < n_taps; ++i) sum += raw[i];
  } else {
    double acc[8];
    for (int j = 0; j < 8; ++j) acc[j] = raw[j];
    int i = 8;
    for (; i < n_taps - n_taps % 8; i += 8)
      for (int j = 0; j < 8; ++j) acc[j] += raw[i + j];
    sum = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
    for (; i < n_taps; ++i) sum += raw[i];
  }
  for (int d = 0; d <= r; ++d) g.w[d] = raw[d + r] / sum;
  const int64_t n = count * (int64_t)H * W;
  if (n == 0) return MEMI_OK;
  const dim3 grid((unsigned)((n + 255) / 256));
  hipStream_t s = (hipStream_t)stream;
  if (in_f64 && out_f64) {
    hipLaunchKernelGGL((k_gauss_pass<double, double, 0>), grid, dim3(256), 0, s,
                       (const double*)in, (double*)tmp, count, H, W, g);
    hipLaunchKernelGGL((k_gauss_pass<double, double, 1>), grid, dim3(256), 0, s,
                       (const double*)tmp, (double*)out, count, H, W, g);
  } else if (in_f64) {
    hipLaunchKernelGGL((k_gauss_pass<double, float, 0>), grid, dim3(256), 0, s,
                       (const double*)in, (float*)tmp, count, H, W, g);
    hipLaunchKernelGGL((k_gauss_pass<float, float, 1>), grid, dim3(256), 0, s,
                       (const float*)tmp, (float*)out, count, H, W, g);
  } else {
    hipLaunchKernelGGL((k_gauss_pass<float, float, 0>), grid, dim3(256), 0, s,
                       (const float*)in, (float*)tmp, count, H, W, g);
    hipLaunchKernelGGL((k_gauss_pass<float, float, 1>), grid, dim3(256), 0, s,
                       (const float*)tmp, (float*)out, count, H, W, g);
  }
  MEMI_CHECK_LAUNCH("k_gauss_pass");
  return MEMI_OK;
}

int memi_hs_derivatives(const float* frames, const int32_t* pairs, int64_t nP, int H, int W,
                        float* fx, float* fy, float* ft, void* stream) {
  MEMI_CHECK_ARG(frames && pairs && fx && fy && ft, "memi_hs_derivatives: null pointer");
  MEMI_CHECK_ARG(nP >= 0 && H >= 1 && W >= 1, "memi_hs_derivatives: bad sizes");
  const int64_t n = nP * (int64_t)H * W;
  if (n == 0) return MEMI_OK;
  hipLaunchKernelGGL(k_hs_derivatives, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, frames, pairs, nP, H, W, fx, fy, ft);
  MEMI_CHECK_LAUNCH("k_hs_derivatives");
  return MEMI_OK;
}

int memi_hs_iterate(const float* fx, const float* fy, const float* ft, int64_t nP, int H, int W,
                    double alpha, int niter, void* U, void* V, int is_f64, void* tmpU,
                    void* tmpV, void* stream) {
  MEMI_CHECK_ARG(fx && fy && ft && U && V && tmpU && tmpV, "memi_hs_iterate: null pointer");
  MEMI_CHECK_ARG(nP >= 0 && H >= 1 && W >= 1 && niter >= 0, "memi_hs_iterate: bad sizes");
  MEMI_CHECK_ARG(tmpU != U && tmpV != V && tmpU != tmpV && U != V,
                 "memi_hs_iterate: U, V, tmpU, tmpV must be distinct");
  if (nP == 0 || niter == 0) return MEMI_OK;
  hipStream_t s = (hipStream_t)stream;
  // numpy adds the Python float alpha**2 to a float32 array as float32
  const float alpha2 = (float)(alpha * alpha);
  int launches, step;
  HsTiling t{};
  int cols = 0;                      // columns per lane of the strip kernel (float64)
  if (is_f64) {
    // the shape and tile counts of least cost: cells computed per iteration, halos included
    // (one column per lane: a tenth more per cell), plus, per launch, the pixels' traffic (44 B
    // at ~8 B per CU cycle, about 18 cells' worth of issue)
    double best = 0.0;
    for (int c = 1; c <= 2; ++c) {
      const int cap_x = 64 * c, cap_y = kHsWaves * hs_strip_rows(c);
      const int nx0 = (W + cap_x - 1) / cap_x, ny0 = (H + cap_y - 1) / cap_y;
      for (int nx = nx0; nx <= nx0 + 2 + nx0 / 4; ++nx)
        for (int ny = ny0; ny <= ny0 + 3 + ny0 / 4; ++ny) {
          const int R = std::min(hs_halo(W, cap_x, nx, niter), hs_halo(H, cap_y, ny, niter));
          if (R < 1) continue;
          const int l = (niter + R - 1) / R;
          const double cost = (c == 1 ? 1.1 : 1.0) * nx * ny * cap_x * cap_y * niter +
                              18.0 * l * H * W;
          if (cols == 0 || cost < best) {
            best = cost;
            cols = c;
            const int h = (niter + l - 1) / l;           // the iterations spread evenly
            t.nx = nx;
            t.ny = ny;
            t.halo = nx * ny == 1 ? 0 : h;
            t.ow = cap_x - 2 * h;
            t.oh = cap_y - 2 * h;
          }
        }
    }
    step = t.halo ? t.halo : niter;
  } else {
    t.nx = (W + kHsTile - 1) / kHsTile;
    t.ny = (H + kHsTile - 1) / kHsTile;
    step = kHsHalo;
  }
  launches = (niter + step - 1) / step;
  const int64_t ntiles = (int64_t)t.nx * t.ny;
  MEMI_CHECK_ARG(nP * ntiles < 0x7fffffffLL, "memi_hs_iterate: too many tiles");
  const size_t bytes = (size_t)nP * H * W * (is_f64 ? 8 : 4);
  // ping-pong so that the last launch writes U, V (one launch of whole images works in place)
  const bool in_place = is_f64 && ntiles == 1;
  void* cur_u = U;
  void* cur_v = V;
  void* nxt_u = in_place ? U : tmpU;
  void* nxt_v = in_place ? V : tmpV;
  if (!in_place && launches % 2) {
    if (hipMemcpyAsync(tmpU, U, bytes, hipMemcpyDeviceToDevice, s) != hipSuccess ||
        hipMemcpyAsync(tmpV, V, bytes, hipMemcpyDeviceToDevice, s) != hipSuccess) {
      set_error("memi_hs_iterate: copy failed");
      return MEMI_ELAUNCH;
    }
    std::swap(cur_u, nxt_u);
    std::swap(cur_v, nxt_v);
  }
  const dim3 grid((unsigned)(nP * ntiles));
  for (int l = 0, done = 0; l < launches; ++l) {
    const int it = std::min(step, niter - done);
    if (is_f64) {
      const dim3 block(kHsWaves * 64);
      const double *ui = (const double*)cur_u, *vi = (const double*)cur_v;
      double *uo = (double*)nxt_u, *vo = (double*)nxt_v;
      if (cols == 1)
        hipLaunchKernelGGL((k_hs_strips<1, hs_strip_rows(1)>), grid, block, 0, s, fx, fy, ft, H,
                           W, t, alpha2, it, ui, vi, uo, vo);
      else
        hipLaunchKernelGGL((k_hs_strips<2, hs_strip_rows(2)>), grid, block, 0, s, fx, fy, ft, H,
                           W, t, alpha2, it, ui, vi, uo, vo);
      MEMI_CHECK_LAUNCH("k_hs_strips");
    } else {
      hipLaunchKernelGGL((k_hs_iterate<kHsTile, kHsHalo, kHsThreads>), grid,
                         dim3(kHsThreads), 0, s, fx, fy, ft, H, W, t.nx, (int)ntiles, alpha2, it,
                         (const float*)cur_u, (const float*)cur_v, (float*)nxt_u,
                         (float*)nxt_v);
      MEMI_CHECK_LAUNCH("k_hs_iterate");
    }
    std::swap(cur_u, nxt_u);
    std::swap(cur_v, nxt_v);
    done += it;
  }
  return MEMI_OK;
}

int memi_flow_sum(const void* U, const void* V, int is_f64, int64_t nmov, int A, int64_t hw,
                  int from_zero, double* vx, double* vy, double* orient, double* mag,
                  double* orient_rev, void* stream) {
  MEMI_CHECK_ARG(U && V && vx && vy, "memi_flow_sum: null pointer");
  MEMI_CHECK_ARG(nmov >= 0 && A >= 1 && hw >= 1, "memi_flow_sum: bad sizes");
  const int64_t n = nmov * hw;
  if (n == 0) return MEMI_OK;
  const dim3 grid((unsigned)((n + 255) / 256));
  if (is_f64)
    hipLaunchKernelGGL(k_flow_sum<double>, grid, dim3(256), 0, (hipStream_t)stream,
                       (const double*)U, (const double*)V, nmov, A, hw, from_zero, vx, vy,
                       orient, mag, orient_rev);
  else
    hipLaunchKernelGGL(k_flow_sum<float>, grid, dim3(256), 0, (hipStream_t)stream,
                       (const float*)U, (const float*)V, nmov, A, hw, from_zero, vx, vy, orient,
                       mag, orient_rev);
  MEMI_CHECK_LAUNCH("k_flow_sum");
  return MEMI_OK;
}

}  // extern "C"
