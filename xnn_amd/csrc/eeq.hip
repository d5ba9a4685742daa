// The real-space part of the large-system EEQ operator (gfx950, float64).
//
// The large regime of the EEQ charges (common/models/eeq.py:170-397, the operator of
// eeq_charges_large, eeq.py:664) splits the Coulomb interaction of the charge
// distributions with an Ewald parameter alpha: the screened kernel
//   K_ij(r) = [erf(gamma_ij r) - erf(alpha r)] / r,  gamma_ij = (a_i^2 + a_j^2)^(-1/2),
// summed over every lattice image within the real-space cutoff (an atom's own images
// included, r > 0), and a reciprocal sum that the host forms from structure factors.
// A molecule takes alpha = 0 and the single image: K = erf(gamma r) / r.
//
// xnn_eeq_real_matrix forms R_ij = sum_n K_ij(|pos_j + n cell - pos_i|) as a dense (N, N)
// float64 matrix (symmetric): one thread per (i, j), the images of the pair in a window
// taken from its fractional coordinates and the cell's interplanar spacings (every image
// within the cutoff lies in it). With 288 GB of HBM the dense matrix is the MI355X form up
// to ~10^5 atoms: it is formed once per evaluation and factorized on the device.
//
// xnn_eeq_real_grad forms the derivatives of S = sum_ij u_i R_ij(pos, cell) w_j: with
// d = pos_j + n cell - pos_i and K' = dK/dr,
//   dS/dpos_k = -sum_{j,n} (u_k w_j + u_j w_k) K'(r) d / r,
//   dS/dcell = sum_k sum_{j,n} u_k w_j K'(r) n (x) d / r   (per-atom rows, summed by the caller),
// one wave per atom k, lanes over j, a fixed butterfly: bitwise reproducible.
// xnn_eeq_real_grad_pairs forms the same over unordered pairs (up to 56,000 atoms).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "common.h"
#include "device.h"
#include "fp64.h"

namespace xnn {

struct EeqCell {
  double a[9];    // rows, bohr
  double inv[9];  // inverse, f = d @ inv
  double reach[3];  // cutoff / interplanar spacing per axis (0: not periodic)
  int periodic;
};

// the window of image offsets n_a for fractional difference f_a: |f_a + n_a| <= reach_a
__device__ inline void image_range(double f, double reach, int& lo, int& hi) {
  lo = (int)ceil(-reach - f);
  hi = (int)floor(reach - f);
}

// erf(gam r) - erf(alpha r) is evaluated as erfc(alpha r) - erfc(gam r), without the
// cancellation of two values near one; erfc(gam r) < 4e-20 for gam r >= 6.5, where it is
// dropped (most pairs of a long real-space range: one error function instead of two).
__device__ inline double screened(double r, double gam, double alpha) {
  if (alpha > 0.0) {
    const double x = gam * r;
    return (erfc(alpha * r) - (x < 6.5 ? erfc(x) : 0.0)) / r;
  }
  return erf(gam * r) / r;
}

// the same from r^2 and 1 / r
__device__ inline double screened_inv(double r2, double ir, double gam, double alpha) {
  const double r = r2 * ir;
  if (alpha > 0.0) {
    const double x = gam * r;
    return (erfc(alpha * r) - (x < 6.5 ? erfc(x) : 0.0)) * ir;
  }
  return erf(gam * r) * ir;
}

// dK/dr of the screened kernel
__device__ inline double screened_slope(double r, double gam, double alpha, double K) {
  constexpr double two_over_sqrt_pi = 1.1283791670955126;
  double g = gam * exp(-gam * gam * r * r);
  if (alpha > 0.0) g -= alpha * exp(-alpha * alpha * r * r);
  return (two_over_sqrt_pi * g - K) / r;
}

// calls fn(dx, dy, dz, n0, n1, n2) for every image n of a pair within distance^2 cut2,
// given the fractional difference f of its two atoms and the per-axis window reach (the
// image offsets with |f_a + n_a| <= reach_a hold every image within the range): f is
// wrapped to [-1/2, 1/2] first and the wrap folded into n. The zero vector (an atom and
// itself) is skipped.
template <typename Fn>
__device__ inline void for_images_frac(const EeqCell& C, const double* reach, double f0,
                                       double f1, double f2, double cut2, Fn&& fn) {
  double f[3] = {f0, f1, f2};
  int w[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    w[c] = (int)rint(f[c]);
    f[c] -= w[c];
  }
  int lo[3], hi[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) image_range(f[c], reach[c], lo[c], hi[c]);
  for (int n0 = lo[0]; n0 <= hi[0]; ++n0)
    for (int n1 = lo[1]; n1 <= hi[1]; ++n1)
      for (int n2 = lo[2]; n2 <= hi[2]; ++n2) {
        const double g0 = f[0] + n0, g1 = f[1] + n1, g2 = f[2] + n2;
        const double dx = g0 * C.a[0] + g1 * C.a[3] + g2 * C.a[6];
        const double dy = g0 * C.a[1] + g1 * C.a[4] + g2 * C.a[7];
        const double dz = g0 * C.a[2] + g1 * C.a[5] + g2 * C.a[8];
        const double r2 = dx * dx + dy * dy + dz * dz;
        if (r2 <= cut2 && r2 > 1e-20) fn(dx, dy, dz, n0 - w[0], n1 - w[1], n2 - w[2]);
      }
}

__device__ inline void to_frac(const EeqCell& C, double dx, double dy, double dz, double* f) {
#pragma unroll
  for (int c = 0; c < 3; ++c) f[c] = dx * C.inv[c] + dy * C.inv[3 + c] + dz * C.inv[6 + c];
}

// calls fn(dx, dy, dz, n0, n1, n2) for every image of the pair (i -> j) within the cutoff
template <typename Fn>
__device__ inline void for_images(const EeqCell& C, double dx0, double dy0, double dz0,
                                  double cut2, bool same, Fn&& fn) {
  if (!C.periodic) {
    const double r2 = dx0 * dx0 + dy0 * dy0 + dz0 * dz0;
    if (!same && r2 <= cut2) fn(dx0, dy0, dz0, 0, 0, 0);
    return;
  }
  double f[3];
  to_frac(C, dx0, dy0, dz0, f);
  for_images_frac(C, C.reach, f[0], f[1], f[2], cut2, fn);
}

// 16 x 16 tiles of the lower block triangle (the upper tiles return at once): each entry
// summed over its images, a tile below the diagonal also stored transposed through LDS, so
// the matrix is symmetric to the bit and half of its entries are summed.
__global__ __launch_bounds__(256) void eeq_real_matrix_kernel(
    const double* __restrict__ pos, int64_t n, EeqCell C, const double* __restrict__ rad,
    double alpha, double cut2, double* __restrict__ R) {
  __shared__ double tile[16][17];
  if (blockIdx.x > blockIdx.y) return;            // uniform: mirrored from below
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  const int64_t j = (int64_t)blockIdx.x * 16 + tx;
  const int64_t i = (int64_t)blockIdx.y * 16 + ty;
  double sum = 0.0;
  if (i < n && j < n) {
    const double ai = rad[i], aj = rad[j];
    const double gam = 1.0 / sqrt(ai * ai + aj * aj);
    for_images(C, pos[3 * j] - pos[3 * i], pos[3 * j + 1] - pos[3 * i + 1],
               pos[3 * j + 2] - pos[3 * i + 2], cut2, i == j,
               [&](double dx, double dy, double dz, int, int, int) {
                 sum += screened(sqrt(dx * dx + dy * dy + dz * dz), gam, alpha);
               });
    R[i * n + j] = sum;
  }
  if (blockIdx.x == blockIdx.y) return;           // uniform: a diagonal tile is whole
  tile[ty][tx] = sum;
  __syncthreads();
  const int64_t it = (int64_t)blockIdx.x * 16 + ty, jt = (int64_t)blockIdx.y * 16 + tx;
  if (it < n && jt < n) R[it * n + jt] = tile[tx][ty];
}

__global__ __launch_bounds__(256) void eeq_real_grad_kernel(
    const double* __restrict__ pos, int64_t n, EeqCell C, const double* __restrict__ rad,
    double alpha, double cut2, const double* __restrict__ u, const double* __restrict__ w,
    double* __restrict__ grad_pos, double* __restrict__ cell_partial) {
  const int lane = threadIdx.x % kWave;
  const int64_t k = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
  if (k >= n) return;
  const double pk0 = pos[3 * k], pk1 = pos[3 * k + 1], pk2 = pos[3 * k + 2];
  const double ak = rad[k], uk = u[k], wk = w[k];
  double g[3] = {0.0, 0.0, 0.0};
  double c[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  const bool want_cell = cell_partial != nullptr;
  for (int64_t j = lane; j < n; j += kWave) {
    const double aj = rad[j];
    const double gam = 1.0 / sqrt(ak * ak + aj * aj);
    const double sym = uk * w[j] + u[j] * wk, own = uk * w[j];
    for_images(C, pos[3 * j] - pk0, pos[3 * j + 1] - pk1, pos[3 * j + 2] - pk2, cut2, j == k,
               [&](double dx, double dy, double dz, int n0, int n1, int n2) {
                 const double r = sqrt(dx * dx + dy * dy + dz * dz);
                 const double K = screened(r, gam, alpha);
                 const double s = screened_slope(r, gam, alpha, K) / r;
                 g[0] -= sym * s * dx;
                 g[1] -= sym * s * dy;
                 g[2] -= sym * s * dz;
                 if (want_cell) {
                   const double t = own * s;
                   c[0] += t * n0 * dx; c[1] += t * n0 * dy; c[2] += t * n0 * dz;
                   c[3] += t * n1 * dx; c[4] += t * n1 * dy; c[5] += t * n1 * dz;
                   c[6] += t * n2 * dx; c[7] += t * n2 * dy; c[8] += t * n2 * dz;
                 }
               });
  }
#pragma unroll
  for (int m = kWave / 2; m > 0; m >>= 1) {
#pragma unroll
    for (int q = 0; q < 3; ++q) g[q] += __shfl_xor(g[q], m, kWave);
    if (want_cell) {
#pragma unroll
      for (int q = 0; q < 9; ++q) c[q] += __shfl_xor(c[q], m, kWave);
    }
  }
  if (lane == 0) {
#pragma unroll
    for (int q = 0; q < 3; ++q) grad_pos[3 * k + q] = g[q];
    if (want_cell) {
#pragma unroll
      for (int q = 0; q < 9; ++q) cell_partial[9 * k + q] = c[q];
    }
  }
}

// The same derivatives over unordered pairs: the lower 64 x 64 tiles, a block a tile, four
// waves of sixteen rows i each, lanes over the columns j. A pair's term goes to its column in
// the lane's registers (the waves' shares added through LDS) and to its row by a butterfly over
// the wave; both are written per tile, part[slot][atom], slots 0 .. T: an atom of tile I gets
// its rows from tiles (I, J), slot J, its columns from (I', I), slot I', those of its own tile
// in slot T; eeq_real_grad_sum_kernel adds the slots in order. The cell's sum is a row of nine
// per block. For the far pairs (gamma r >= 7, where gamma's terms are below 1e-21) one error
// function and one exponential remain, and 1/r is a refined estimate instead of three divisions.
// 5,000 atoms, 2.7 images a pair: 0.93 ms, where the directed kernel takes 2.07.
constexpr int kGradTile = 64;
// part is (T + 1) x 3 N doubles, 1.2 GB at the most; beyond that the directed kernel
constexpr int64_t kGradMaxAtoms = 56000;

__global__ __launch_bounds__(256) void eeq_real_grad_tiles_kernel(
    const double* __restrict__ pos, int64_t n, EeqCell C, const double* __restrict__ rad,
    double alpha, double cut2, const double* __restrict__ u, const double* __restrict__ w,
    int64_t n_tiles, bool want_cell, double* __restrict__ part, double* __restrict__ cell_rows) {
  __shared__ double sg[4][3][kGradTile], sc[4][9];
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const int64_t b = blockIdx.x;
  int64_t ti = (int64_t)((sqrt(8.0 * (double)b + 1.0) - 1.0) * 0.5);
  while (ti * (ti + 1) / 2 > b) --ti;
  while ((ti + 1) * (ti + 2) / 2 <= b) ++ti;
  const int64_t tj = b - ti * (ti + 1) / 2;
  const int64_t j = tj * kGradTile + lane, jc = min(j, n - 1);
  const double xj = pos[3 * jc], yj = pos[3 * jc + 1], zj = pos[3 * jc + 2];
  const double aj = rad[jc], uj = u[jc], wj = w[jc];
  double g[3] = {0.0, 0.0, 0.0}, c[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  constexpr double two_over_sqrt_pi = 1.1283791670955126;
  for (int q = 0; q < kGradTile / 4; ++q) {
    const int64_t i = ti * kGradTile + wv * (kGradTile / 4) + q;
    if (i >= n) break;                                    // uniform in the wave
    double f[3] = {0.0, 0.0, 0.0};
    if (j <= i && j < n) {
      const double ai = rad[i], gam = rsq_nr(fma(ai, ai, aj * aj));
      const double sym = j == i ? u[i] * w[i] : u[i] * wj + uj * w[i];
      for_images(C, xj - pos[3 * i], yj - pos[3 * i + 1], zj - pos[3 * i + 2], cut2, j == i,
                 [&](double dx, double dy, double dz, int n0, int n1, int n2) {
                   const double r2 = dx * dx + dy * dy + dz * dz, ir = rsq_nr(r2);
                   const double x = gam * (r2 * ir);
                   double e = x < 7.0 ? gam * exp(-x * x) : 0.0;
                   if (alpha > 0.0) e -= alpha * exp(-(alpha * alpha) * r2);
                   const double K = screened_inv(r2, ir, gam, alpha);
                   const double s = sym * ((two_over_sqrt_pi * e - K) * ir) * ir;
                   const double px = s * dx, py = s * dy, pz = s * dz;
                   f[0] += px;
                   f[1] += py;
                   f[2] += pz;
                   if (want_cell) {
                     c[0] = fma(n0, px, c[0]); c[1] = fma(n0, py, c[1]); c[2] = fma(n0, pz, c[2]);
                     c[3] = fma(n1, px, c[3]); c[4] = fma(n1, py, c[4]); c[5] = fma(n1, pz, c[5]);
                     c[6] = fma(n2, px, c[6]); c[7] = fma(n2, py, c[7]); c[8] = fma(n2, pz, c[8]);
                   }
                 });
      if (j == i) f[0] = f[1] = f[2] = 0.0;               // an atom and its images: no force
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) g[a] += f[a];
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1)
#pragma unroll
      for (int a = 0; a < 3; ++a) f[a] += __shfl_xor(f[a], m, kWave);
    if (lane == 0)
#pragma unroll
      for (int a = 0; a < 3; ++a) part[(tj * n + i) * 3 + a] = -f[a];
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) sg[wv][a][lane] = g[a];
  if (want_cell) {
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1)
#pragma unroll
      for (int q = 0; q < 9; ++q) c[q] += __shfl_xor(c[q], m, kWave);
    if (lane == 0)
#pragma unroll
      for (int q = 0; q < 9; ++q) sc[wv][q] = c[q];
  }
  __syncthreads();
  if (wv < 3 && j < n)                                    // wave a: component a
    part[((ti == tj ? n_tiles : ti) * n + j) * 3 + wv] =
        (sg[0][wv][lane] + sg[1][wv][lane]) + (sg[2][wv][lane] + sg[3][wv][lane]);
  if (want_cell && wv == 3 && lane < 9)
    cell_rows[b * 9 + lane] = (sc[0][lane] + sc[1][lane]) + (sc[2][lane] + sc[3][lane]);
}

__global__ __launch_bounds__(256) void eeq_real_grad_sum_kernel(const double* __restrict__ part,
                                                                int64_t slots, int64_t m,
                                                                double* __restrict__ out) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= m) return;
  double s = 0.0;
#pragma unroll 8
  for (int64_t q = 0; q < slots; ++q) s += part[q * m + e];
  out[e] = s;
}

// out[q] = the sum of rows[b][q], a block per component, strided shares added in order
__global__ __launch_bounds__(256) void eeq_cell_sum_kernel(const double* __restrict__ rows,
                                                           int64_t n_rows, double* __restrict__ out) {
  __shared__ double s[256];
  double v = 0.0;
#pragma unroll 4
  for (int64_t b = threadIdx.x; b < n_rows; b += 256) v += rows[b * 9 + blockIdx.x];
  s[threadIdx.x] = v;
  for (int m = 128; m > 0; m >>= 1) {
    __syncthreads();
    if ((int)threadIdx.x < m) s[threadIdx.x] += s[threadIdx.x + m];
  }
  if (threadIdx.x == 0) out[blockIdx.x] = s[0];
}

static int64_t grad_tiles(int64_t n) { return (n + kGradTile - 1) / kGradTile; }

// ------------------------------------------------------------------ matrix-free product
// out = R v for one or two right-hand sides (the conjugate-gradient regime): R is never
// stored. Atoms come in tiles of kApplyTile consecutive indices; block (i tile, split)
// takes the i tile, one atom per thread, against the j tiles of its split, staged in LDS
// (fractional coordinates, width, v), and writes its partial sums; the splits are added
// in a fixed order afterwards (bitwise reproducible). With tile bounds (center, radius of
// a sphere holding the tile's atoms, in the coordinates of pos), a j tile is skipped when
// no lattice image of it comes within the cutoff of the i tile: ordered along space (the
// cell list of the caller), most tiles of a large cell are skipped.
constexpr int kApplyTile = 256;
constexpr int kApplyBlocks = 2048;   // target blocks per launch (8 per CU)

__device__ inline bool eeq_tiles_meet(const EeqCell& C, const double* __restrict__ tiles,
                                      int64_t ti, int64_t tj, double cutoff) {
  const double* a = tiles + 4 * ti;
  const double* b = tiles + 4 * tj;
  const double R = cutoff + a[3] + b[3];
  const double dx = b[0] - a[0], dy = b[1] - a[1], dz = b[2] - a[2];
  if (!C.periodic) return dx * dx + dy * dy + dz * dz <= R * R;
  double f[3], reach[3];
  to_frac(C, dx, dy, dz, f);
#pragma unroll
  for (int c = 0; c < 3; ++c) reach[c] = C.reach[c] * (R / cutoff) + 1e-12;
  bool hit = dx * dx + dy * dy + dz * dz <= R * R;   // the zero image, which the walk skips
  for_images_frac(C, reach, f[0], f[1], f[2], R * R,
                  [&](double, double, double, int, int, int) { hit = true; });
  return hit;
}

template <int NRHS>
__global__ __launch_bounds__(kApplyTile) void eeq_real_apply_kernel(
    const double* __restrict__ pos, int64_t n, EeqCell C, const double* __restrict__ rad,
    double alpha, double cutoff, const double* __restrict__ tiles,
    const double* __restrict__ v, int64_t tiles_per_split, double* __restrict__ part) {
  __shared__ double sp[3][kApplyTile], sa[kApplyTile], sv[NRHS][kApplyTile];
  const int64_t ti = blockIdx.x, split = blockIdx.y;
  const int64_t n_tiles = (n + kApplyTile - 1) / kApplyTile;
  const int64_t i = ti * kApplyTile + threadIdx.x;
  const bool vi = i < n;
  const int64_t ic = vi ? i : 0;
  double pi[3];
  if (C.periodic) {
    to_frac(C, pos[3 * ic], pos[3 * ic + 1], pos[3 * ic + 2], pi);
  } else {
#pragma unroll
    for (int c = 0; c < 3; ++c) pi[c] = pos[3 * ic + c];
  }
  const double ai2 = rad[ic] * rad[ic];
  const double cut2 = cutoff * cutoff;
  double acc[NRHS];
#pragma unroll
  for (int r = 0; r < NRHS; ++r) acc[r] = 0.0;
  const int64_t t0 = split * tiles_per_split;
  const int64_t t1 = t0 + tiles_per_split < n_tiles ? t0 + tiles_per_split : n_tiles;
  for (int64_t tj = t0; tj < t1; ++tj) {
    if (tiles != nullptr && !eeq_tiles_meet(C, tiles, ti, tj, cutoff)) continue;  // uniform
    const int64_t j0 = tj * kApplyTile;
    const int cnt = (int)(n - j0 < kApplyTile ? n - j0 : kApplyTile);
    __syncthreads();
    if ((int)threadIdx.x < cnt) {
      const int64_t j = j0 + threadIdx.x;
      double pj[3];
      if (C.periodic) {
        to_frac(C, pos[3 * j], pos[3 * j + 1], pos[3 * j + 2], pj);
      } else {
#pragma unroll
        for (int c = 0; c < 3; ++c) pj[c] = pos[3 * j + c];
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) sp[c][threadIdx.x] = pj[c];
      sa[threadIdx.x] = rad[j] * rad[j];
#pragma unroll
      for (int r = 0; r < NRHS; ++r) sv[r][threadIdx.x] = v[j * NRHS + r];
    }
    __syncthreads();
    if (!vi) continue;
    for (int q = 0; q < cnt; ++q) {
      // refined hardware reciprocal square roots (about an ulp) instead of the IEEE square
      // roots and divisions: the kernel value only needs float64 accuracy, not rounding
      const double gam = rsq_nr(ai2 + sa[q]);
      double k = 0.0;
      const auto add = [&](double dx, double dy, double dz, int, int, int) {
        const double r2 = dx * dx + dy * dy + dz * dz;
        k += screened_inv(r2, rsq_nr(r2), gam, alpha);
      };
      if (C.periodic) {
        for_images_frac(C, C.reach, sp[0][q] - pi[0], sp[1][q] - pi[1], sp[2][q] - pi[2], cut2,
                        add);
      } else if (j0 + q != i) {
        const double dx = sp[0][q] - pi[0], dy = sp[1][q] - pi[1], dz = sp[2][q] - pi[2];
        if (dx * dx + dy * dy + dz * dz <= cut2) add(dx, dy, dz, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < NRHS; ++r) acc[r] = fma(k, sv[r][q], acc[r]);
    }
  }
  if (vi) {
#pragma unroll
    for (int r = 0; r < NRHS; ++r) part[(split * n + i) * NRHS + r] = acc[r];
  }
}

// out[k] = sum over the splits of part[s][k], in split order
__global__ __launch_bounds__(256) void eeq_sum_splits_kernel(const double* __restrict__ part,
                                                             int64_t splits, int64_t m,
                                                             double* __restrict__ out) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= m) return;
  double s = 0.0;
  for (int64_t q = 0; q < splits; ++q) s += part[q * m + k];
  out[k] = s;
}

// ------------------------------------------------------------------ stored product
// The same product from the real-space matrix evaluated once (the conjugate-gradient regime
// multiplies it some fifty times): its lower 128 x 128 tiles, packed. Of each row of a tile
// that has an image within the cutoff, a bit per column and the values of the set ones (8.2
// bytes per unordered pair in reach), each read once per product and used for both of its
// atoms. A block takes a tile, its waves 32 rows each, a lane the columns l and l + 64; the
// wave holds its 64 half rows' bits and places in its lanes and hands them out as scalars.
// The column sums stay in the lane, the row sums of 32 (row, side) pairs at a time go
// through a reduce-scatter over the wave (31 exchanges instead of six butterfly steps a
// row). Both are written per tile and summed per row by eeq_tiles_sum_kernel in tile order
// (bitwise reproducible). Bound by reading the values: two columns at 24,000 atoms and 60
// bohr (1.3 GB) take 331 us = 4.0 TB/s and 35 us of sums, where evaluating the 5.8e8 pairs
// takes 4,800 us; forming the values takes 4,000 us once.
constexpr int kStoreTile = 128;

// the lane's place among the lanes of mask below it
__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// v[l] kept from the halving over lane bit M: lanes with the bit take hi, the others lo, each
// adding its partner's value of the same slot
template <int M>
__device__ __forceinline__ double halve_lanes(double lo, double hi, int lane) {
  const bool up = lane & M;
  const double keep = up ? hi : lo;
  const double give = up ? lo : hi;
  if constexpr (M == 8) {
    const int a = __builtin_amdgcn_mov_dpp(__double2loint(give), 0x128, 0xF, 0xF, false);
    const int b = __builtin_amdgcn_mov_dpp(__double2hiint(give), 0x128, 0xF, 0xF, false);
    return keep + __hiloint2double(b, a);
  } else {
    return keep + xor_lanes<M>(give);
  }
}

// the two halves (M = 32) or the 16-lane rows of each half (M = 16): lo stays with the lanes
// without the bit, hi with the others (row-swap permutes, no selects)
template <int M>
__device__ __forceinline__ double halve_swap(double lo, double hi) {
  const unsigned a0 = (unsigned)__double2loint(lo), a1 = (unsigned)__double2hiint(lo);
  const unsigned b0 = (unsigned)__double2loint(hi), b1 = (unsigned)__double2hiint(hi);
  const auto x = M == 32 ? __builtin_amdgcn_permlane32_swap(a0, b0, false, false)
                         : __builtin_amdgcn_permlane16_swap(a0, b0, false, false);
  const auto y = M == 32 ? __builtin_amdgcn_permlane32_swap(a1, b1, false, false)
                         : __builtin_amdgcn_permlane16_swap(a1, b1, false, false);
  return __hiloint2double((int)y[0], (int)x[0]) + __hiloint2double((int)y[1], (int)x[1]);
}

// the wave-wide sums of 32 per-lane values: lanes 2k and 2k + 1 return the total of value k
__device__ __forceinline__ double reduce_scatter32(double (&p)[32], int lane) {
#pragma unroll
  for (int k = 0; k < 16; ++k) p[k] = halve_swap<32>(p[k], p[k + 16]);
#pragma unroll
  for (int k = 0; k < 8; ++k) p[k] = halve_swap<16>(p[k], p[k + 8]);
#pragma unroll
  for (int k = 0; k < 4; ++k) p[k] = halve_lanes<8>(p[k], p[k + 4], lane);
#pragma unroll
  for (int k = 0; k < 2; ++k) p[k] = halve_lanes<4>(p[k], p[k + 2], lane);
  p[0] = halve_lanes<2>(p[0], p[1], lane);
  return p[0] + xor_lanes<1>(p[0]);
}

template <int NRHS>
__global__ __launch_bounds__(256) void eeq_tiles_apply_kernel(
    const double* __restrict__ values, const int32_t* __restrict__ tile_ij,
    const uint64_t* __restrict__ mask, const uint32_t* __restrict__ off,
    const int64_t* __restrict__ base, int64_t n, const double* __restrict__ v,
    double* __restrict__ part) {
  constexpr int kRows = 32 / NRHS;                 // rows per reduce-scatter
  __shared__ double sv[kStoreTile * NRHS];         // v of the row block
  __shared__ double sc[4][kStoreTile * NRHS];      // the waves' column sums
  const int64_t id = blockIdx.x;
  const int64_t I = tile_ij[2 * id], J = tile_ij[2 * id + 1];
  const int lane = threadIdx.x % kWave, w = wave_in_block();
  // half row 64 w + lane of the tile: row 32 w + lane / 2, columns 64 (lane % 2) + 0..63
  const int64_t half_row = id * (2 * kStoreTile) + 64 * w + lane;
  const uint64_t my_mask = mask[half_row];
  const int my_off = (int)off[half_row];
  const int mask_lo = (int)(uint32_t)my_mask, mask_hi = (int)(uint32_t)(my_mask >> 32);
  const double* vals = values + base[id];
  // a wave without values loads none: a tile without any may start at the end of them all
  const bool any = __ballot(my_mask != 0) != 0;    // uniform in the wave
  for (int k = threadIdx.x; k < kStoreTile * NRHS; k += 256) {
    const int64_t at = I * kStoreTile * NRHS + k;
    sv[k] = at < n * NRHS ? v[at] : 0.0;
  }
  double vj[2][NRHS], col[2][NRHS];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < NRHS; ++r) {
      const int64_t j = J * kStoreTile + lane + 64 * h;
      vj[h][r] = j < n ? v[j * NRHS + r] : 0.0;
      col[h][r] = 0.0;
    }
  __syncthreads();
  double* out = part + id * (2 * kStoreTile * NRHS);
  if (!any)
    for (int k = lane; k < 32 * NRHS; k += kWave) out[32 * w * NRHS + k] = 0.0;
  for (int b = 0; any && b < 32; b += kRows) {
    double a[kRows][2];
#pragma unroll
    for (int q = 0; q < kRows; ++q)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = 2 * (b + q) + h;
        const uint64_t m = (uint64_t)(uint32_t)__builtin_amdgcn_readlane(mask_lo, k) |
                           (uint64_t)(uint32_t)__builtin_amdgcn_readlane(mask_hi, k) << 32;
        const int at = __builtin_amdgcn_readlane(my_off, k) + (int)lanes_below(m);
        // every lane loads (an unset column the tile's first value), so that no load waits
        // for a branch
        const double x = vals[(m >> lane) & 1 ? at : 0];
        a[q][h] = (m >> lane) & 1 ? x : 0.0;
      }
    double p[32];
#pragma unroll
    for (int q = 0; q < kRows; ++q)
#pragma unroll
      for (int r = 0; r < NRHS; ++r) {
        p[q * NRHS + r] = fma(a[q][1], vj[1][r], a[q][0] * vj[0][r]);
        const double vi = sv[(32 * w + b + q) * NRHS + r];
        col[0][r] = fma(a[q][0], vi, col[0][r]);
        col[1][r] = fma(a[q][1], vi, col[1][r]);
      }
    const double t = reduce_scatter32(p, lane);
    if ((lane & 1) == 0) out[(32 * w + b) * NRHS + lane / 2] = t;
  }
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < NRHS; ++r) sc[w][(lane + 64 * h) * NRHS + r] = col[h][r];
  __syncthreads();
  for (int k = threadIdx.x; k < kStoreTile * NRHS; k += 256)
    out[kStoreTile * NRHS + k] = ((sc[0][k] + sc[1][k]) + sc[2][k]) + sc[3][k];
}

// out of row block I: the row sums of its tiles (I, J <= I) and the column sums of the tiles
// (K > I, I), 1024 / (128 NRHS) partial sums over the blocks taken in turn, added in order
template <int NRHS>
__global__ __launch_bounds__(1024) void eeq_tiles_sum_kernel(const double* __restrict__ part,
                                                             const int32_t* __restrict__ index,
                                                             int64_t n, int64_t nt,
                                                             double* __restrict__ out) {
  constexpr int kW = kStoreTile * NRHS, kGroups = 1024 / kW, kAhead = 8;
  __shared__ double sums[kGroups][kW];
  const int64_t I = blockIdx.x;
  const int k = threadIdx.x % kW, g = threadIdx.x / kW;
  double s = 0.0;
  for (int64_t K0 = g; K0 < nt; K0 += kGroups * kAhead) {
    double x[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int64_t K = K0 + u * kGroups;
      const int64_t hi = K > I ? K : I, lo = K > I ? I : K;
      const int64_t id = K < nt ? (int64_t)index[hi * nt + lo] : -1;
      x[u] = id >= 0 ? part[(id * 2 + (K > I ? 1 : 0)) * kW + k] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) s += x[u];
  }
  sums[g][k] = s;
  __syncthreads();
  if (g != 0) return;
#pragma unroll
  for (int q = 1; q < kGroups; ++q) s += sums[q][k];
  const int64_t at = I * kW + k;
  if (at < n * NRHS) out[at] = s;
}

// flags[I * nt + J] = 1 for the lower tiles with an image within the cutoff, else 0
__global__ __launch_bounds__(256) void eeq_store_meet_kernel(EeqCell C, const double* __restrict__ tiles,
                                                             int64_t nt, double cutoff,
                                                             int32_t* __restrict__ flags) {
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (k >= nt * nt) return;
  const int64_t I = k / nt, J = k % nt;
  flags[k] = J <= I && (tiles == nullptr || eeq_tiles_meet(C, tiles, I, J, cutoff)) ? 1 : 0;
}

// One tile: which columns of each row have an image within the cutoff (FILL = false: the
// bits, each half row's place and the number of values), and their entries of
// eeq_real_matrix_kernel (FILL). A wave takes 32 rows, a lane the columns l and l + 64.
template <bool FILL>
__global__ __launch_bounds__(256) void eeq_store_kernel(
    const double* __restrict__ pos, int64_t n, EeqCell C, const double* __restrict__ rad,
    double alpha, double cut2, const int32_t* __restrict__ tile_ij, uint64_t* __restrict__ mask,
    uint32_t* __restrict__ off, int64_t* __restrict__ count, const int64_t* __restrict__ base,
    double* __restrict__ values) {
  __shared__ double sp[3][kStoreTile], sa[kStoreTile];
  __shared__ uint32_t place[kStoreTile * 2], wave_total[4];
  const int64_t id = blockIdx.x, i0 = (int64_t)tile_ij[2 * id] * kStoreTile;
  const int64_t j0 = (int64_t)tile_ij[2 * id + 1] * kStoreTile;
  const int lane = threadIdx.x % kWave, w = wave_in_block();
  if (threadIdx.x < kStoreTile) {
    const int c = threadIdx.x;
    const int64_t i = i0 + c < n ? i0 + c : 0;
    double p[3] = {pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]};
    if (C.periodic) to_frac(C, pos[3 * i], pos[3 * i + 1], pos[3 * i + 2], p);
#pragma unroll
    for (int q = 0; q < 3; ++q) sp[q][c] = p[q];
    sa[c] = FILL ? rad[i] * rad[i] : 0.0;
  }
  double pj[2][3], aj2[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int64_t j = j0 + lane + 64 * h, jc = j < n ? j : 0;
#pragma unroll
    for (int q = 0; q < 3; ++q) pj[h][q] = pos[3 * jc + q];
    if (C.periodic) to_frac(C, pos[3 * jc], pos[3 * jc + 1], pos[3 * jc + 2], pj[h]);
    aj2[h] = FILL ? rad[jc] * rad[jc] : 0.0;
  }
  __syncthreads();
  uint32_t total = 0;
  for (int q = w * 32; q < w * 32 + 32; ++q)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t j = j0 + lane + 64 * h, row = (id * kStoreTile + q) * 2 + h;
      const double d0 = pj[h][0] - sp[0][q], d1 = pj[h][1] - sp[1][q], d2 = pj[h][2] - sp[2][q];
      const bool pair = j < n && i0 + q < n;
      double k = 0.0;
      bool near = false;
      const double gam = FILL ? rsq_nr(sa[q] + aj2[h]) : 0.0;
      const auto add = [&](double dx, double dy, double dz, int, int, int) {
        near = true;
        if constexpr (FILL) {
          const double r2 = dx * dx + dy * dy + dz * dz;
          k += screened_inv(r2, rsq_nr(r2), gam, alpha);
        }
      };
      if (pair && C.periodic) {
        for_images_frac(C, C.reach, d0, d1, d2, cut2, add);
      } else if (pair && i0 + q != j && d0 * d0 + d1 * d1 + d2 * d2 <= cut2) {
        add(d0, d1, d2, 0, 0, 0);
      }
      if constexpr (FILL) {
        const uint64_t m = mask[row];
        if ((m >> lane) & 1) values[base[id] + off[row] + lanes_below(m)] = k;
      } else {
        const uint64_t m = __ballot(near);
        if (lane == 0) {
          mask[row] = m;
          place[q * 2 + h] = total;
        }
        total += __popcll(m);
      }
    }
  if constexpr (!FILL) {
    if (lane == 0) wave_total[w] = total;
    __syncthreads();
    const int k = threadIdx.x;                      // one half row a thread
    uint32_t before = 0;
    for (int x = 0; x < k / 64; ++x) before += wave_total[x];
    off[id * (2 * kStoreTile) + k] = before + place[k];
    if (k == 0) count[id] = (int64_t)wave_total[0] + wave_total[1] + wave_total[2] + wave_total[3];
  }
}

// ------------------------------------------------------------------ molecules
// The dense regime's charges of a batch of molecules (d4.py:593-606, 682-723): per molecule
// [A 1; 1^T 0] [q; mu] = [x; Q] with A_ij = erf(gamma_ij r_ij) / r_ij, A_ii = diag_i, built and
// eliminated with partial pivoting in one workgroup's LDS (m = n + 1 rows of m + 1 values,
// the last the right-hand side; rows stay in place, `row` is their order). The adjoint solve
// of the backward (the matrix is symmetric) eliminates again, which is cheaper than
// keeping factors; then dL/dx = lambda and, a thread per atom,
// dL/dpos_k = -sum_j (lambda_k q_j + lambda_j q_k) K'(r) (pos_k - pos_j) / r.
// Bound by the elimination's two barriers a row: 32 molecules of 21 atoms take 37 us forward and
// 51 us backward, where a solve call and its backward per molecule (2,900 launches and a
// synchronization each) took 22 ms of the energy's and forces' 24 ms.
constexpr int kMolThreads = 256;
constexpr int kMolMaxAtoms = 128;   // 129 rows of 131 doubles: 135 KB of the CU's 160 KB

template <bool BWD>
__global__ __launch_bounds__(kMolThreads) void eeq_molecule_kernel(
    const double* __restrict__ pos, int64_t n_nodes, const int64_t* __restrict__ node_ptr,
    const int32_t* __restrict__ ids, const double* __restrict__ rad,
    const double* __restrict__ diag, const double* __restrict__ rhs,
    const double* __restrict__ total, int max_atoms, const double* __restrict__ q,
    double* __restrict__ out, double* __restrict__ grad_pos, int32_t* __restrict__ info) {
  extern __shared__ double mol_lds[];
  __shared__ double sp[3][kMolMaxAtoms], srad[kMolMaxAtoms], sx[kMolMaxAtoms + 1];
  __shared__ double sq[BWD ? kMolMaxAtoms : 1];
  __shared__ int row[kMolMaxAtoms + 1];
  const int64_t b = ids != nullptr ? ids[blockIdx.x] : blockIdx.x;
  const int64_t a0 = min<int64_t>(max<int64_t>(node_ptr[b], 0), n_nodes);
  const int64_t a1 = min<int64_t>(max<int64_t>(node_ptr[b + 1], a0), n_nodes);
  const int n = (int)(a1 - a0), m = n + 1, t = threadIdx.x;
  if (n == 0 || n > max_atoms) return;              // uniform
  const int ld = (m + 1) | 1;                       // odd: a column's rows in distinct banks
  double* A = mol_lds;
  for (int i = t; i < n; i += kMolThreads) {
#pragma unroll
    for (int c = 0; c < 3; ++c) sp[c][i] = pos[3 * (a0 + i) + c];
    srad[i] = rad[a0 + i];
    if (BWD) sq[i] = q[a0 + i];
  }
  for (int i = t; i < m; i += kMolThreads) row[i] = i;
  __syncthreads();
  for (int e = t; e < m * m; e += kMolThreads) {
    const int i = e / m, j = e % m;
    double v;
    if (i < n && j < n && i != j) {
      const double dx = sp[0][i] - sp[0][j], dy = sp[1][i] - sp[1][j], dz = sp[2][i] - sp[2][j];
      const double r = sqrt(dx * dx + dy * dy + dz * dz);
      v = erf(r / sqrt(srad[i] * srad[i] + srad[j] * srad[j])) / r;
    } else {
      v = i < n && j < n ? diag[a0 + i] : (i == j ? 0.0 : 1.0);
    }
    A[i * ld + j] = v;
  }
  for (int i = t; i < m; i += kMolThreads)
    A[i * ld + m] = i < n ? rhs[a0 + i] : (BWD || total == nullptr ? 0.0 : total[b]);
  __syncthreads();
  const int tx = t % 32, ty = t / 32;
  for (int k = 0; k < m; ++k) {
    if (t < kWave) {                                // the pivot: the largest entry, first of equals
      double best = -1.0;
      int at = k;
      for (int i = k + t; i < m; i += kWave) {
        const double v = fabs(A[row[i] * ld + k]);
        if (v > best) {
          best = v;
          at = i;
        }
      }
#pragma unroll
      for (int o = 1; o < kWave; o <<= 1) {
        const double v = __shfl_xor(best, o, kWave);
        const int w = __shfl_xor(at, o, kWave);
        if (v > best || (v == best && w < at)) {
          best = v;
          at = w;
        }
      }
      if (t == 0) {
        if (best == 0.0) atomicOr(info, 1);
        const int r = row[k];
        row[k] = row[at];
        row[at] = r;
      }
    }
    __syncthreads();
    const double* pk = A + row[k] * ld;
    const double pivot = pk[k];
    for (int i = k + 1 + ty; i < m; i += kMolThreads / 32) {
      double* pi = A + row[i] * ld;
      const double f = pi[k] / pivot;
      for (int j = k + 1 + tx; j <= m; j += 32) pi[j] = fma(-f, pk[j], pi[j]);
    }
    __syncthreads();
  }
  for (int k = m - 1; k >= 0; --k) {
    const double x = A[row[k] * ld + m] / A[row[k] * ld + k];
    if (t == 0) sx[k] = x;
    for (int i = t; i < k; i += kMolThreads)
      A[row[i] * ld + m] = fma(-A[row[i] * ld + k], x, A[row[i] * ld + m]);
    __syncthreads();
  }
  for (int i = t; i < n; i += kMolThreads) {
    out[a0 + i] = sx[i];
    if (BWD) {
      double g[3] = {0.0, 0.0, 0.0};
      for (int j = 0; j < n; ++j) {
        if (j == i) continue;
        const double d[3] = {sp[0][i] - sp[0][j], sp[1][i] - sp[1][j], sp[2][i] - sp[2][j]};
        const double r = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
        const double gam = 1.0 / sqrt(srad[i] * srad[i] + srad[j] * srad[j]);
        const double s = screened_slope(r, gam, 0.0, erf(gam * r) / r) / r;
        const double w = -(sx[i] * sq[j] + sx[j] * sq[i]) * s;
#pragma unroll
        for (int c = 0; c < 3; ++c) g[c] = fma(w, d[c], g[c]);
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) grad_pos[3 * (a0 + i) + c] = g[c];
    }
  }
}

template <bool BWD>
static int launch_molecules(const double* pos, int64_t n_nodes, const int64_t* node_ptr,
                            const int32_t* ids, int64_t n_ids, int64_t max_atoms,
                            const double* rad, const double* diag, const double* rhs,
                            const double* total, const double* q, double* out, double* grad_pos,
                            int32_t* info, hipStream_t s) {
  const int m = (int)max_atoms + 1;
  const size_t lds = sizeof(double) * (size_t)m * ((m + 1) | 1);
  const auto k = eeq_molecule_kernel<BWD>;
  if (lds > 48 * 1024)
    XNN_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(k, dim3((unsigned)n_ids), dim3(kMolThreads), lds, s, pos, n_nodes, node_ptr,
                     ids, rad, diag, rhs, total, (int)max_atoms, q, out, grad_pos, info);
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

static int64_t eeq_apply_splits(int64_t n) {
  const int64_t tiles = (n + kApplyTile - 1) / kApplyTile;
  if (tiles == 0) return 1;
  const int64_t want = (kApplyBlocks + tiles - 1) / tiles;
  return std::max<int64_t>(1, std::min<int64_t>(want, tiles));
}

// host: the cell's inverse and per-axis reach; false for a singular cell
static bool eeq_cell(const double* cell, double cutoff, EeqCell& C) {
  C.periodic = cell != nullptr;
  for (int q = 0; q < 9; ++q) {
    C.a[q] = cell ? cell[q] : 0.0;
    C.inv[q] = 0.0;
  }
  C.reach[0] = C.reach[1] = C.reach[2] = 0.0;
  if (!C.periodic) return true;
  const double* a = C.a;
  const double c00 = a[4] * a[8] - a[5] * a[7], c01 = a[2] * a[7] - a[1] * a[8],
               c02 = a[1] * a[5] - a[2] * a[4];
  const double det = a[0] * c00 + a[3] * c01 + a[6] * c02;
  if (!(std::fabs(det) > 1e-12)) return false;
  const double id = 1.0 / det;
  C.inv[0] = c00 * id;
  C.inv[1] = c01 * id;
  C.inv[2] = c02 * id;
  C.inv[3] = (a[5] * a[6] - a[3] * a[8]) * id;
  C.inv[4] = (a[0] * a[8] - a[2] * a[6]) * id;
  C.inv[5] = (a[2] * a[3] - a[0] * a[5]) * id;
  C.inv[6] = (a[3] * a[7] - a[4] * a[6]) * id;
  C.inv[7] = (a[1] * a[6] - a[0] * a[7]) * id;
  C.inv[8] = (a[0] * a[4] - a[1] * a[3]) * id;
  // interplanar spacing of axis c: 1 / |column c of the inverse|; a little slack so that
  // rounding never drops an image at the cutoff (the r test decides)
  for (int col = 0; col < 3; ++col) {
    const double x = C.inv[col], y = C.inv[3 + col], z = C.inv[6 + col];
    C.reach[col] = cutoff * std::sqrt(x * x + y * y + z * z) * (1.0 + 1e-12) + 1e-12;
  }
  return true;
}

// the image windows stay bounded: at most kMaxReach cell lengths along any axis
constexpr double kMaxReach = 32.0;
static bool eeq_reach_ok(const EeqCell& C, double cutoff) {
  if (!C.periodic) return true;
  if (!std::isfinite(cutoff)) return false;
  return C.reach[0] <= kMaxReach && C.reach[1] <= kMaxReach && C.reach[2] <= kMaxReach;
}


// ------------------------------------------------------------------ factorization
// The blocked right-looking Cholesky factorization of the (symmetric positive definite)
// operator, lower triangle in place, 128 columns at a time: the diagonal block and its
// inverse in one workgroup, the panel below it times the inverse's transpose, and the
// trailing matrix's lower tiles, all on the float64 matrix cores (v_mfma_f64_16x16x4: lane l
// gives A[l % 16][l / 16] and B[l / 16][l % 16] and gets D[4 v + l / 16][l % 16]).
// 5,000 rows: 3.4 ms (40 blocks of 33 us, panels of 16 us, trailing updates of 38 us), where
// vector arithmetic for the block (97 us) and library products for the rest took 6.7 ms.
typedef double doublex4 __attribute__((ext_vector_type(4)));
constexpr int kCholBlock = 128;
constexpr int kCholThreads = 512;
constexpr int kCholT = 16;                                // tile edge
constexpr int kCholTiles = kCholBlock / kCholT;           // 8 tile rows
constexpr int kCholLd = kCholT + 1;                       // odd: a tile's rows in distinct banks
constexpr int kCholTile = kCholT * kCholLd;
constexpr int kCholLower = kCholTiles * (kCholTiles + 1) / 2;

__device__ __forceinline__ double* chol_tile(double* base, int i, int j) {
  return base + (i * (i + 1) / 2 + j) * kCholTile;
}

// acc += A B^T (TRANS) or A B of 16 x 16 tiles of leading dimension kCholLd
template <bool TRANS>
__device__ __forceinline__ doublex4 chol_mfma(const double* A, const double* B, doublex4 acc) {
  const int l = threadIdx.x & (kWave - 1), lo = l & 15, hi = l >> 4;
#pragma unroll
  for (int k = 0; k < kCholT; k += 4) {
    const double a = A[lo * kCholLd + k + hi];
    const double b = TRANS ? B[lo * kCholLd + k + hi] : B[(k + hi) * kCholLd + lo];
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
  }
  return acc;
}

// C -= A B^T (TRANS) or A B; C in place
template <bool TRANS>
__device__ __forceinline__ void chol_subtract(double* C, const double* A, const double* B) {
  const int l = threadIdx.x & (kWave - 1), lo = l & 15, hi = l >> 4;
  const doublex4 p = chol_mfma<TRANS>(A, B, doublex4{0.0, 0.0, 0.0, 0.0});
#pragma unroll
  for (int v = 0; v < 4; ++v) C[(4 * v + hi) * kCholLd + lo] -= p[v];
}

// C = A B^T (TRANS) or A B; C may be one of them
template <bool TRANS>
__device__ __forceinline__ void chol_product(double* C, const double* A, const double* B) {
  const int l = threadIdx.x & (kWave - 1), lo = l & 15, hi = l >> 4;
  const doublex4 p = chol_mfma<TRANS>(A, B, doublex4{0.0, 0.0, 0.0, 0.0});
#pragma unroll
  for (int v = 0; v < 4; ++v) C[(4 * v + hi) * kCholLd + lo] = p[v];
}

// the value of lane C of each row of 16 lanes
template <int C>
__device__ __forceinline__ double row_lane(double v) {
  constexpr int kRowNewBcast = 0x150;
  union {
    double d;
    long long w;
  } u;
  u.d = v;
  u.w = __builtin_amdgcn_update_dpp(u.w, u.w, kRowNewBcast + C, 0xf, 0xf, true);
  return u.d;
}

// 1 / sqrt(d) for a positive normal d: the hardware estimate y and one third-order step,
// y (1 + e / 2 + 3 e^2 / 8) with e = 1 - d y y
__device__ __forceinline__ double refined_rsqrt(double d) {
  const double y = __builtin_amdgcn_rsq(d), e = fma(-d * y, y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

// v[c] -= L_cj v[j] and e[c] -= L_cj e[j] for c = C .. 15, L_cj lane c's v[j]
template <int J, int C>
__device__ __forceinline__ void chol_column(double (&v)[kCholT], double (&e)[kCholT]) {
  if constexpr (C < kCholT) {
    const double m = -row_lane<C>(v[J]);
    v[C] = fma(m, v[J], v[C]);
    e[C] = fma(m, e[J], e[C]);
    chol_column<J, C + 1>(v, e);
  }
}

template <int J>
__device__ __forceinline__ void chol_columns(double (&v)[kCholT], double (&e)[kCholT], int& bad) {
  if constexpr (J < kCholT) {
    const double d = row_lane<J>(v[J]), s = refined_rsqrt(d);
    bad = d > 0.0 && d < INFINITY ? bad : min(bad, J);
    v[J] *= s;
    e[J] *= s;
    chol_column<J, J + 1>(v, e);
    __builtin_amdgcn_sched_barrier(0);                    // or broadcasts pile up and spill
    chol_columns<J + 1>(v, e, bad);
  }
}

// One wave factors a 16 x 16 tile in registers and inverts the factor with the same
// operations: lane i of each 16 holds row i of the tile (v) and column i of what starts as
// the identity (e); step j scales both registers j by 1 / sqrt(pivot) and takes L_cj times
// them from every register c > j, L_cj broadcast from lane c. No barrier and no LDS between
// the 16 steps. Returns the first column whose pivot is not positive and finite, or 16.
__device__ __forceinline__ int chol_factor_tile(double* A, double* inv) {
  const int lo = threadIdx.x & 15;
  double v[kCholT], e[kCholT];
#pragma unroll
  for (int c = 0; c < kCholT; ++c) {
    v[c] = A[lo * kCholLd + c];
    e[c] = c == lo ? 1.0 : 0.0;
  }
  int bad = kCholT;
  chol_columns<0>(v, e, bad);
  // the four lanes of a row write the same values: under a branch the compiler would sink the
  // steps into it, and hold every broadcast until then
#pragma unroll
  for (int c = 0; c < kCholT; ++c) {
    A[lo * kCholLd + c] = c <= lo ? v[c] : 0.0;
    inv[c * kCholLd + lo] = c >= lo ? e[c] : 0.0;
  }
  return bad;
}

// The diagonal block [k0, k0 + b) (leading dimension lda): L in place (the block's upper
// triangle zeroed) and inv = L^-1 (b, b) row-major. The block's 36 lower 16 x 16 tiles and
// the 36 of E, which starts as the identity and ends as L^-1, are in LDS; step p takes the
// factor and inverse of the diagonal tile, then column p of the block (A_ip <- A_ip inv^T)
// and row p of E (E_pj <- inv E_pj), seven products for eight waves, then A_ij -= A_ip A_jp^T
// and E_ij -= A_ip E_pj below. Wave 0 updates and factors the next diagonal tile while the
// other seven do the rest. Rows past b are the identity's. A pivot that is not positive and
// finite stores k0 + its column + 1 into *info if it still holds 0 and leaves the block
// unwritten.
// 33 us: the 128 dependent pivots of wave 0 half of it (4,400 cycles a tile), a quarter the
// reads and writes of one compute unit.
__global__ __launch_bounds__(kCholThreads) void eeq_cholesky_block_kernel(
    double* __restrict__ a, int64_t lda, int64_t k0, int b, double* __restrict__ inv,
    int* __restrict__ info) {
  extern __shared__ double chol_lds[];
  double* A = chol_lds;
  double* E = A + kCholLower * kCholTile;
  __shared__ int s_bad;
  const int t = threadIdx.x, w = t >> 6;
  double* blk = a + k0 * lda + k0;
  // four rows of the block a pass, a tile row's loads before their first use. Loops are kept
  // rolled: the code runs once, and fetching it costs more than its branches
  const int tr = t >> 7, tc = t & 127;
  const int own = (tc >> 4) * kCholTile + tr * kCholLd + (tc & 15);
  if (t == 0) s_bad = kCholBlock;
#pragma unroll 1
  for (int I = 0; I < kCholTiles; ++I) {
    const int at = I * (I + 1) / 2 * kCholTile + own;
    double in[4];
#pragma unroll
    for (int x = 0; x < 4; ++x)
      in[x] = blk[(int64_t)min(kCholT * I + 4 * x + tr, b - 1) * lda +
                  min(tc, min(kCholT * (I + 1), b) - 1)];  // the lower tiles' lines only
    if (tc < kCholT * (I + 1)) {
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int i = kCholT * I + 4 * x + tr;
        A[at + 4 * x * kCholLd] = max(i, tc) < b ? in[x] : (i == tc ? 1.0 : 0.0);
        E[at + 4 * x * kCholLd] = 0.0;
      }
    }
  }
  __syncthreads();
#pragma unroll 1
  for (int p = 0; p < kCholTiles; ++p) {
    if (w == 0) {                                         // tile (p, p), after column p - 1
      double* const N = chol_tile(A, p, p);
      if (p > 0) chol_subtract<true>(N, chol_tile(A, p, p - 1), chol_tile(A, p, p - 1));
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the lanes' stores, then reads
      const int bad = chol_factor_tile(N, chol_tile(E, p, p));
      if (t == 0 && bad < kCholT) s_bad = kCholT * p + bad;
    } else if (p > 0) {
      // the other tiles after column p - 1: row i holds E's tiles j < p and the block's
      // p <= j <= i, i + 1 of them, in the order of the rows without tile (p, p)
      int at = w - 1;
#pragma unroll 1
      for (int i = p; i < kCholTiles; ++i) {
        const int m = i == p ? p : i + 1;
#pragma unroll 1
        for (; at < m; at += kCholThreads / kWave - 1) {
          if (at < p)
            chol_subtract<false>(chol_tile(E, i, at), chol_tile(A, i, p - 1), chol_tile(E, p - 1, at));
          else
            chol_subtract<true>(chol_tile(A, i, at), chol_tile(A, i, p - 1), chol_tile(A, at, p - 1));
        }
        at -= m;
      }
    }
    __syncthreads();
    if (s_bad < kCholBlock) {                             // uniform
      if (t == 0 && *info == 0) *info = (int)(k0 + s_bad + 1);
      return;
    }
    double* const D = chol_tile(E, p, p);
    if (w < p)                                            // E_pj, j = w
      chol_product<false>(chol_tile(E, p, w), D, chol_tile(E, p, w));
    else if (w + 1 < kCholTiles)                          // A_ip, i = w + 1
      chol_product<true>(chol_tile(A, w + 1, p), chol_tile(A, w + 1, p), D);
    __syncthreads();
  }
#pragma unroll 1
  for (int I = 0; I < kCholTiles; ++I) {
    const int at = I * (I + 1) / 2 * kCholTile + own;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int i = kCholT * I + 4 * x + tr;
      if (i >= b || tc >= b) continue;
      blk[(int64_t)i * lda + tc] = tc <= i ? A[at + 4 * x * kCholLd] : 0.0;
      inv[i * b + tc] = tc <= i ? E[at + 4 * x * kCholLd] : 0.0;
    }
  }
}

// The panel below a full diagonal block, in place: rows [r0, n), columns [k0, k0 + 128):
// P <- P inv^T. A workgroup holds 32 rows in LDS and walks the inverse 32 rows (32 columns of
// the result) at a time; it writes only rows that it alone reads. inv is lower triangular:
// columns c .. c + 16 take the first c + 16 terms.
constexpr int kPanelRows = 32;
constexpr int kPanelLd = kCholBlock + 2;                  // 4-word steps: 2 lanes a bank, the least

__global__ __launch_bounds__(256) void eeq_cholesky_panel_kernel(double* __restrict__ a, int64_t n,
                                                                 int64_t k0, int64_t r0,
                                                                 const double* __restrict__ inv) {
  __shared__ double P[kPanelRows * kPanelLd], V[kPanelRows * kPanelLd];
  const int t = threadIdx.x, l = t & (kWave - 1), lo = l & 15, hi = l >> 4, w = t >> 6;
  const int tr = t >> 7, tc = t & 127;
  const int64_t row0 = r0 + (int64_t)blockIdx.x * kPanelRows;
  double in[kPanelRows / 2], nx[kPanelRows / 2];
#pragma unroll
  for (int r = 0; r < kPanelRows; r += 2) {               // rows past n: the last row again, unstored
    in[r / 2] = a[min<int64_t>(row0 + r + tr, n - 1) * n + k0 + tc];
    nx[r / 2] = inv[(r + tr) * kCholBlock + tc];
  }
#pragma unroll
  for (int r = 0; r < kPanelRows; r += 2) P[(r + tr) * kPanelLd + tc] = in[r / 2];
  const int mt = w & 1, nt = w >> 1;                      // the wave's 16 x 16 part of 32 x 32
  for (int c0 = 0; c0 < kCholBlock; c0 += 32) {
#pragma unroll
    for (int r = 0; r < 32; r += 2) V[(r + tr) * kPanelLd + tc] = nx[r / 2];
    __syncthreads();
    if (c0 + 32 < kCholBlock) {                           // the next 32 rows, in flight meanwhile
#pragma unroll
      for (int r = 0; r < 32; r += 2) nx[r / 2] = inv[(c0 + 32 + r + tr) * kCholBlock + tc];
    }
    doublex4 acc{0.0, 0.0, 0.0, 0.0};
    const double* pa = P + (16 * mt + lo) * kPanelLd + hi;
    const double* pb = V + (16 * nt + lo) * kPanelLd + hi;
    const int kend = c0 + 16 * nt + 16;
#pragma unroll 4
    for (int k = 0; k < kend; k += 4)
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(pa[k], pb[k], acc, 0, 0, 0);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t i = row0 + 16 * mt + 4 * v + hi;
      if (i < n) a[i * n + k0 + c0 + 16 * nt + lo] = acc[v];
    }
    __syncthreads();
  }
}

// The trailing matrix's 64 x 64 tiles on and below the diagonal: C_ij -= P_i P_j^T with the
// panel P = rows [r0, n) of columns [k0, k0 + 128), in two chunks of 64 columns through LDS
// (68 KB: two workgroups a compute unit, one loads while the other multiplies). Four waves of
// 32 x 32. A tile is 512 matrix instructions of 64 cycles on four SIMDs, 3.4 us, against 128
// KB of panel from L2. 5,000 rows' 40,000 tiles take 1.48 ms, 0.55 of it the matrix cores'; the
// rest is the wait for each tile's first loads and the last, part-filled round of a launch.
constexpr int kTrailTile = 64;
constexpr int kTrailLd = kTrailTile + 2;

__global__ __launch_bounds__(256) void eeq_cholesky_trail_kernel(double* __restrict__ a, int64_t n,
                                                                 int64_t k0, int64_t r0) {
  __shared__ double P[kTrailTile * kTrailLd], Q[kTrailTile * kTrailLd];
  const int t = threadIdx.x, l = t & (kWave - 1), lo = l & 15, hi = l >> 4, w = t >> 6;
  // tile (ti, tj), tj <= ti, of the row-major lower triangle
  const int64_t g = blockIdx.x;
  int64_t ti = (int64_t)((sqrt(8.0 * (double)g + 1.0) - 1.0) * 0.5);
  while (ti * (ti + 1) / 2 > g) --ti;
  while ((ti + 1) * (ti + 2) / 2 <= g) ++ti;
  const int64_t tj = g - ti * (ti + 1) / 2;
  const int64_t i0 = r0 + ti * kTrailTile, j0 = r0 + tj * kTrailTile;
  const int mr = 32 * (w & 1), nc = 32 * (w >> 1);
  doublex4 acc[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t i = i0 + mr + 16 * x + 4 * v + hi, j = j0 + nc + 16 * y + lo;
        acc[x][y][v] = a[min(i, n - 1) * n + min(j, n - 1)];
      }
  double pi[kTrailTile / 4], pj[kTrailTile / 4];
  const auto load = [&](int c0) {                         // rows past n: the last row again, unstored
#pragma unroll
    for (int r = 0; r < kTrailTile; r += 4) {
      pi[r / 4] = a[min(i0 + r + w, n - 1) * n + k0 + c0 + l];
      pj[r / 4] = a[min(j0 + r + w, n - 1) * n + k0 + c0 + l];
    }
  };
  load(0);
#pragma unroll 1
  for (int c0 = 0; c0 < kCholBlock; c0 += kTrailTile) {
#pragma unroll
    for (int r = 0; r < kTrailTile; r += 4) {
      P[(r + w) * kTrailLd + l] = -pi[r / 4];
      Q[(r + w) * kTrailLd + l] = pj[r / 4];
    }
    if (c0 + kTrailTile < kCholBlock) load(c0 + kTrailTile);   // in flight during the products
    __syncthreads();
#pragma unroll 4
    for (int k = 0; k < kTrailTile; k += 4) {
      double pa[2], pb[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        pa[x] = P[(mr + 16 * x + lo) * kTrailLd + k + hi];
        pb[x] = Q[(nc + 16 * x + lo) * kTrailLd + k + hi];
      }
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
          acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(pa[x], pb[y], acc[x][y], 0, 0, 0);
    }
    __syncthreads();
  }
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t i = i0 + mr + 16 * x + 4 * v + hi, j = j0 + nc + 16 * y + lo;
        if (i < n && j < n) a[i * n + j] = acc[x][y][v];
      }
}

static int launch_cholesky_block(double* matrix, int64_t n, int64_t k0, int b, double* inv,
                                 int* info, hipStream_t s) {
  constexpr size_t lds = sizeof(double) * 2 * kCholLower * kCholTile;
  static_assert(lds + 64 <= 160 * 1024, "a compute unit's LDS");
  XNN_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(eeq_cholesky_block_kernel),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(eeq_cholesky_block_kernel, dim3(1), dim3(kCholThreads), lds, s, matrix, n, k0, b,
                     inv, info);
  return XNN_OK;
}

// ---------------------------------------------------------------- solves with the factor
// (L L^T) X = B with L from eeq_cholesky_block_kernel and the inverses of its diagonal
// blocks (block j: rows [128 j, 128 j + b_j), inverse at inv + 128 * 128 j, row stride
// b_j), X (n, NRHS) row-major. Forward L Y = B walks the blocks down, backward L^T X = Y
// up, one launch per block. Launch k: every workgroup solves block k from its residual
// rows with the block's inverse (forward y = inv r, backward x = inv^T r; a 128 x 128
// product, repeated per workgroup rather than waiting for one), workgroup 0 stores it,
// and every row still to come takes away the block's contribution (forward: r_i -= L[i,
// k0:k0 + b_k] y_k, 32 rows a workgroup; backward: r_i -= L[k0:k0 + b_k, i]^T x_k for i <
// k0, 64 rows a workgroup). Everything a launch reads is loaded first, unconditionally (past
// an edge the last valid entry, dropped by a select), so the chain of a launch is one memory
// latency and the two products. The solution goes to another array than the residual rows
// the launch reads (forward: residual in X, solution in the work array; backward the
// reverse), so no workgroup reads a row another one rewrites. Sums in a fixed order.
// 40 blocks of 5,000 rows: 7.5 us a forward and 6.4 us a backward launch of one column (8.5
// and 6.4 of two), where loads behind bounds tests, one latency each, took 11.4 and 13.8.
constexpr int kTrsvBlock = kCholBlock;
constexpr int kTrsvThreads = 512;
constexpr int kTrsvGroups = kTrsvThreads / kTrsvBlock;    // 4 threads per row or column of a block
constexpr int kTrsvPer = kTrsvBlock / kTrsvGroups;        // entries each of them takes
constexpr int kTrsvFwdRows = 32;      // rows per workgroup (forward): four a wave
constexpr int kTrsvBwdRows = 64;      // rows per workgroup (backward)
constexpr int kTrsvWaves = kTrsvThreads / kWave;
constexpr int kTrsvFwdBatch = kTrsvFwdRows / kTrsvWaves;  // rows of L a wave takes (forward)
constexpr int kTrsvBwdBatch = kTrsvBlock / kTrsvWaves;    // and rows of the block (backward)

__device__ __forceinline__ double wave_sum_xor(double v) {
#pragma unroll
  for (int m = kWave / 2; m > 0; m >>= 1) v += __shfl_xor(v, m, kWave);
  return v;
}

template <int NRHS>
__global__ __launch_bounds__(kTrsvThreads) void eeq_trsv_forward_kernel(
    const double* __restrict__ L, int64_t n, const double* __restrict__ inv, int k,
    double* __restrict__ res, double* __restrict__ sol) {
  extern __shared__ double trsv_lds[];                    // the inverse, rows of 129
  __shared__ double rs[kTrsvBlock][NRHS];                 // block k's residual
  __shared__ double xs[kTrsvBlock][NRHS];                 // its solution
  constexpr int kLd = kTrsvBlock + 1;
  const int t = threadIdx.x, lane = t & (kWave - 1), wv = t >> 6;
  const int64_t k0 = (int64_t)k * kTrsvBlock;
  const int bk = (int)(n - k0 < kTrsvBlock ? n - k0 : kTrsvBlock);
  const double* ib = inv + (int64_t)k * kTrsvBlock * kTrsvBlock;
  const int g = t / kTrsvBlock, c = t % kTrsvBlock;
  double m[kTrsvPer], v0[kTrsvFwdBatch], v1[kTrsvFwdBatch], old[kTrsvFwdBatch][NRHS], r0[NRHS];
#pragma unroll
  for (int r = 0; r < NRHS; ++r) r0[r] = res[(k0 + min(c, bk - 1)) * NRHS + r];
#pragma unroll
  for (int q = 0; q < kTrsvPer; ++q)
    m[q] = ib[min(kTrsvGroups * q + g, bk - 1) * bk + min(c, bk - 1)];
  const int64_t i0 = k0 + bk + (int64_t)blockIdx.x * kTrsvFwdRows + wv * kTrsvFwdBatch;
#pragma unroll
  for (int q = 0; q < kTrsvFwdBatch; ++q) {
    const int64_t i = min(i0 + q, n - 1);
    v0[q] = L[i * n + k0 + min(lane, bk - 1)];
    v1[q] = L[i * n + k0 + min(lane + kWave, bk - 1)];
#pragma unroll
    for (int r = 0; r < NRHS; ++r) old[q][r] = res[i * NRHS + r];
  }
  if (g == 0) {
#pragma unroll
    for (int r = 0; r < NRHS; ++r) rs[c][r] = c < bk ? r0[r] : 0.0;
  }
#pragma unroll
  for (int q = 0; q < kTrsvPer; ++q) trsv_lds[(kTrsvGroups * q + g) * kLd + c] = m[q];
  __syncthreads();
  {  // four threads an entry, over entries h, h + 4, ...
    const int i = t / kTrsvGroups, h = t % kTrsvGroups;
    double s[NRHS];
#pragma unroll
    for (int r = 0; r < NRHS; ++r) s[r] = 0.0;
#pragma unroll
    for (int q = 0; q < kTrsvPer; ++q) {
      const int cc = kTrsvGroups * q + h;
      const double l = cc <= i ? trsv_lds[i * kLd + cc] : 0.0;
#pragma unroll
      for (int r = 0; r < NRHS; ++r) s[r] = fma(l, rs[cc][r], s[r]);
    }
#pragma unroll
    for (int r = 0; r < NRHS; ++r) {
      s[r] += __shfl_xor(s[r], 1, kWave);
      s[r] += __shfl_xor(s[r], 2, kWave);
      if (h == 0) xs[i][r] = i < bk ? s[r] : 0.0;
    }
  }
  __syncthreads();
  if (blockIdx.x == 0)
    for (int i = t; i < bk * NRHS; i += kTrsvThreads) sol[k0 * NRHS + i] = (&xs[0][0])[i];
#pragma unroll
  for (int q = 0; q < kTrsvFwdBatch; ++q) {
#pragma unroll
    for (int r = 0; r < NRHS; ++r) {
      const double a = lane < bk ? v0[q] * xs[lane][r] : 0.0;
      const double sr = wave_sum_xor(lane + kWave < bk ? fma(v1[q], xs[lane + kWave][r], a) : a);
      if (lane == 0 && i0 + q < n) res[(i0 + q) * NRHS + r] = old[q][r] - sr;
    }
  }
}

template <int NRHS>
__global__ __launch_bounds__(kTrsvThreads) void eeq_trsv_backward_kernel(
    const double* __restrict__ L, int64_t n, const double* __restrict__ inv, int k,
    double* __restrict__ res, double* __restrict__ sol) {
  __shared__ double rs[kTrsvBlock][NRHS];                 // block k's residual
  __shared__ double xs[kTrsvBlock][NRHS];                 // its solution
  __shared__ double part[kTrsvGroups][kTrsvBlock][NRHS];
  __shared__ double upd[kTrsvWaves][kTrsvBwdRows][NRHS];
  const int t = threadIdx.x, lane = t & (kWave - 1), wv = t >> 6;
  const int64_t k0 = (int64_t)k * kTrsvBlock;
  const int bk = (int)(n - k0 < kTrsvBlock ? n - k0 : kTrsvBlock);
  const double* ib = inv + (int64_t)k * kTrsvBlock * kTrsvBlock;
  const int g = t / kTrsvBlock, c = t % kTrsvBlock;
  double m[kTrsvPer], l[kTrsvBwdBatch], old[NRHS], r0[NRHS];
#pragma unroll
  for (int r = 0; r < NRHS; ++r) r0[r] = res[(k0 + min(c, bk - 1)) * NRHS + r];
#pragma unroll
  for (int q = 0; q < kTrsvPer; ++q)
    m[q] = ib[min(kTrsvGroups * q + g, bk - 1) * bk + min(c, bk - 1)];
  const int64_t i = (int64_t)blockIdx.x * kTrsvBwdRows + lane;   // < k0 or past the rows
  const int64_t ic = min(i, n - 1);
#pragma unroll
  for (int q = 0; q < kTrsvBwdBatch; ++q)
    l[q] = L[(k0 + min(wv * kTrsvBwdBatch + q, bk - 1)) * n + ic];
#pragma unroll
  for (int r = 0; r < NRHS; ++r) old[r] = res[ic * NRHS + r];
  if (g == 0) {
#pragma unroll
    for (int r = 0; r < NRHS; ++r) rs[c][r] = c < bk ? r0[r] : 0.0;
  }
  __syncthreads();
  double s[NRHS];
#pragma unroll
  for (int r = 0; r < NRHS; ++r) s[r] = 0.0;
#pragma unroll
  for (int q = 0; q < kTrsvPer; ++q) {                    // rows below or at the entry's own
    const int row = kTrsvGroups * q + g;
    const double e = row >= c && row < bk ? m[q] : 0.0;
#pragma unroll
    for (int r = 0; r < NRHS; ++r) s[r] = fma(e, rs[row][r], s[r]);
  }
#pragma unroll
  for (int r = 0; r < NRHS; ++r) part[g][c][r] = s[r];
  __syncthreads();
  for (int e = t; e < kTrsvBlock * NRHS; e += kTrsvThreads) {
    double x = 0.0;
#pragma unroll
    for (int h = 0; h < kTrsvGroups; ++h) x += (&part[h][0][0])[e];
    (&xs[0][0])[e] = e < bk * NRHS ? x : 0.0;
    if (blockIdx.x == 0 && e < bk * NRHS) sol[k0 * NRHS + e] = x;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < NRHS; ++r) s[r] = 0.0;
#pragma unroll
  for (int q = 0; q < kTrsvBwdBatch; ++q) {
    const int row = wv * kTrsvBwdBatch + q;
    const double e = row < bk ? l[q] : 0.0;
#pragma unroll
    for (int r = 0; r < NRHS; ++r) s[r] = fma(e, xs[row][r], s[r]);
  }
#pragma unroll
  for (int r = 0; r < NRHS; ++r) upd[wv][lane][r] = s[r];
  __syncthreads();
  if (wv == 0 && i < k0) {
#pragma unroll
    for (int r = 0; r < NRHS; ++r) {
      double x = 0.0;
#pragma unroll
      for (int h = 0; h < kTrsvWaves; ++h) x += upd[h][lane][r];
      res[i * NRHS + r] = old[r] - x;
    }
  }
}

template <int NRHS>
static int launch_trsv(const double* factor, int64_t n, const double* inv_blocks, double* x,
                       double* work, hipStream_t s) {
  const int nb = (int)((n + kTrsvBlock - 1) / kTrsvBlock);
  constexpr size_t lds = sizeof(double) * kTrsvBlock * (kTrsvBlock + 1);
  const auto fwd = eeq_trsv_forward_kernel<NRHS>;
  XNN_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(fwd),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  for (int k = 0; k < nb; ++k) {          // forward: residual in x, solution into work
    const int64_t after = n - std::min<int64_t>(n, (int64_t)(k + 1) * kTrsvBlock);
    const unsigned grid = (unsigned)std::max<int64_t>(1, (after + kTrsvFwdRows - 1) / kTrsvFwdRows);
    hipLaunchKernelGGL(fwd, dim3(grid), dim3(kTrsvThreads), lds, s, factor, n, inv_blocks, k, x, work);
  }
  for (int k = nb - 1; k >= 0; --k) {     // backward: residual in work, solution into x
    const int64_t before = (int64_t)k * kTrsvBlock;
    const unsigned grid = (unsigned)std::max<int64_t>(1, (before + kTrsvBwdRows - 1) / kTrsvBwdRows);
    hipLaunchKernelGGL(eeq_trsv_backward_kernel<NRHS>, dim3(grid), dim3(kTrsvThreads), 0, s, factor, n,
                       inv_blocks, k, work, x);
  }
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

}  // namespace xnn

using namespace xnn;

extern "C" {

int xnn_eeq_real_matrix(const double* pos, int64_t n_nodes, const double* cell,
                        const double* rad, double alpha, double cutoff, double* matrix,
                        xnn_stream_t stream) {
  XNN_REQUIRE(n_nodes >= 0, "negative size");
  if (n_nodes == 0) return XNN_OK;
  XNN_REQUIRE(pos && rad && matrix, "NULL input or output");
  XNN_REQUIRE(n_nodes <= (int64_t(1) << 20), "at most 2^20 atoms");
  XNN_REQUIRE(cutoff > 0.0 && alpha >= 0.0, "cutoff must be positive, alpha non-negative");
  XNN_REQUIRE(cell != nullptr || alpha == 0.0, "a molecule takes alpha = 0");
  EeqCell C;
  XNN_REQUIRE(eeq_cell(cell, cutoff, C), "singular cell");
  XNN_REQUIRE(eeq_reach_ok(C, cutoff), "the real-space range spans more than %g cells",
              kMaxReach);
  const dim3 grid((unsigned)((n_nodes + 15) / 16), (unsigned)((n_nodes + 15) / 16));
  hipLaunchKernelGGL(eeq_real_matrix_kernel, grid, dim3(256), 0, as_hip(stream), pos, n_nodes, C,
                     rad, alpha, cutoff * cutoff, matrix);
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

int xnn_eeq_real_grad(const double* pos, int64_t n_nodes, const double* cell, const double* rad,
                      double alpha, double cutoff, const double* u, const double* w,
                      double* grad_pos, double* cell_partial, xnn_stream_t stream) {
  XNN_REQUIRE(n_nodes >= 0, "negative size");
  if (n_nodes == 0) return XNN_OK;
  XNN_REQUIRE(pos && rad && u && w && grad_pos, "NULL input or output");
  XNN_REQUIRE(cutoff > 0.0 && alpha >= 0.0, "cutoff must be positive, alpha non-negative");
  XNN_REQUIRE(cell != nullptr || (alpha == 0.0 && cell_partial == nullptr),
              "a molecule takes alpha = 0 and has no cell gradient");
  EeqCell C;
  XNN_REQUIRE(eeq_cell(cell, cutoff, C), "singular cell");
  XNN_REQUIRE(eeq_reach_ok(C, cutoff), "the real-space range spans more than %g cells",
              kMaxReach);
  hipLaunchKernelGGL(eeq_real_grad_kernel, dim3((unsigned)grid_1d(n_nodes, 4)), dim3(256), 0,
                     as_hip(stream), pos, n_nodes, C, rad, alpha, cutoff * cutoff, u, w, grad_pos,
                     cell_partial);
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

int xnn_eeq_real_grad_pairs_work_size(int64_t n_nodes, size_t* bytes) {
  XNN_REQUIRE(n_nodes >= 0 && bytes != nullptr, "negative size or NULL result");
  const int64_t t = grad_tiles(n_nodes);
  *bytes = n_nodes > kGradMaxAtoms
               ? 0 : sizeof(double) * (size_t)((t + 1) * 3 * n_nodes + 9 * (t * (t + 1) / 2));
  return XNN_OK;
}

int xnn_eeq_real_grad_pairs(const double* pos, int64_t n_nodes, const double* cell,
                            const double* rad, double alpha, double cutoff, const double* u,
                            const double* w, double* grad_pos, double* grad_cell, void* work,
                            size_t work_bytes, xnn_stream_t stream) {
  XNN_REQUIRE(n_nodes >= 1 && n_nodes <= kGradMaxAtoms, "1 to %lld atoms", (long long)kGradMaxAtoms);
  XNN_REQUIRE(pos && rad && u && w && grad_pos && work, "NULL input, output or work");
  XNN_REQUIRE(cutoff > 0.0 && alpha >= 0.0, "cutoff must be positive, alpha non-negative");
  XNN_REQUIRE(cell != nullptr || (alpha == 0.0 && grad_cell == nullptr),
              "a molecule takes alpha = 0 and has no cell gradient");
  EeqCell C;
  XNN_REQUIRE(eeq_cell(cell, cutoff, C), "singular cell");
  XNN_REQUIRE(eeq_reach_ok(C, cutoff), "the real-space range spans more than %g cells",
              kMaxReach);
  size_t need = 0;
  (void)xnn_eeq_real_grad_pairs_work_size(n_nodes, &need);
  XNN_REQUIRE(work_bytes >= need, "work too small");
  const int64_t t = grad_tiles(n_nodes), blocks = t * (t + 1) / 2;
  double* part = static_cast<double*>(work);
  double* rows = part + (t + 1) * 3 * n_nodes;
  hipStream_t s = as_hip(stream);
  hipLaunchKernelGGL(eeq_real_grad_tiles_kernel, dim3((unsigned)blocks), dim3(256), 0, s, pos, n_nodes,
                     C, rad, alpha, cutoff * cutoff, u, w, t, grad_cell != nullptr, part, rows);
  hipLaunchKernelGGL(eeq_real_grad_sum_kernel, dim3((unsigned)grid_1d(3 * n_nodes, 256)), dim3(256), 0, s,
                     part, t + 1, 3 * n_nodes, grad_pos);
  if (grad_cell != nullptr)
    hipLaunchKernelGGL(eeq_cell_sum_kernel, dim3(9), dim3(256), 0, s, rows, blocks, grad_cell);
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

int xnn_eeq_real_apply_work_size(int64_t n_nodes, int32_t nrhs, size_t* bytes) {
  XNN_REQUIRE(n_nodes >= 0 && bytes != nullptr, "negative size or NULL output");
  XNN_REQUIRE(nrhs == 1 || nrhs == 2, "one or two right-hand sides (got %d)", (int)nrhs);
  *bytes = sizeof(double) * (size_t)std::max<int64_t>(eeq_apply_splits(n_nodes) * n_nodes * nrhs, 1);
  return XNN_OK;
}

int xnn_eeq_real_apply(const double* pos, int64_t n_nodes, const double* cell, const double* rad,
                       double alpha, double cutoff, const double* tiles, const double* v,
                       int32_t nrhs, double* out, void* work, size_t work_bytes,
                       xnn_stream_t stream) {
  XNN_REQUIRE(n_nodes >= 0, "negative size");
  XNN_REQUIRE(nrhs == 1 || nrhs == 2, "one or two right-hand sides (got %d)", (int)nrhs);
  if (n_nodes == 0) return XNN_OK;
  XNN_REQUIRE(pos && rad && v && out && work, "NULL input, output or workspace");
  XNN_REQUIRE(n_nodes <= (int64_t(1) << 26), "at most 2^26 atoms");
  XNN_REQUIRE(cutoff > 0.0 && alpha >= 0.0, "cutoff must be positive, alpha non-negative");
  XNN_REQUIRE(cell != nullptr || alpha == 0.0, "a molecule takes alpha = 0");
  const int64_t splits = eeq_apply_splits(n_nodes);
  XNN_REQUIRE(work_bytes >= sizeof(double) * (size_t)(splits * n_nodes * nrhs),
              "workspace too small");
  EeqCell C;
  XNN_REQUIRE(eeq_cell(cell, cutoff, C), "singular cell");
  XNN_REQUIRE(eeq_reach_ok(C, cutoff), "the real-space range spans more than %g cells",
              kMaxReach);
  const int64_t n_tiles = (n_nodes + kApplyTile - 1) / kApplyTile;
  const int64_t per = (n_tiles + splits - 1) / splits;
  const dim3 grid((unsigned)n_tiles, (unsigned)splits);
  hipStream_t s = as_hip(stream);
  double* part = static_cast<double*>(work);
  if (nrhs == 1)
    hipLaunchKernelGGL(eeq_real_apply_kernel<1>, grid, dim3(kApplyTile), 0, s, pos, n_nodes, C,
                       rad, alpha, cutoff, tiles, v, per, part);
  else
    hipLaunchKernelGGL(eeq_real_apply_kernel<2>, grid, dim3(kApplyTile), 0, s, pos, n_nodes, C,
                       rad, alpha, cutoff, tiles, v, per, part);
  XNN_LAUNCH_CHECK();
  const int64_t m = n_nodes * nrhs;
  hipLaunchKernelGGL(eeq_sum_splits_kernel, dim3((unsigned)grid_1d(m, 256)), dim3(256), 0, s, part,
                     splits, m, out);
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

int xnn_eeq_store_meet(const double* tiles, int64_t n_nodes, const double* cell, double cutoff,
                       int32_t* flags, xnn_stream_t stream) {
  XNN_REQUIRE(n_nodes >= 0, "negative size");
  if (n_nodes == 0) return XNN_OK;
  XNN_REQUIRE(flags != nullptr && cutoff > 0.0, "NULL flags or a cutoff that is not positive");
  XNN_REQUIRE(n_nodes <= (int64_t(1) << 21), "at most 2^21 atoms");
  EeqCell C;
  XNN_REQUIRE(eeq_cell(cell, cutoff, C), "singular cell");
  XNN_REQUIRE(eeq_reach_ok(C, cutoff), "the real-space range spans more than %g cells",
              kMaxReach);
  const int64_t nt = (n_nodes + kStoreTile - 1) / kStoreTile;
  hipLaunchKernelGGL(eeq_store_meet_kernel, dim3((unsigned)grid_1d(nt * nt, 256)), dim3(256), 0,
                     as_hip(stream), C, tiles, nt, cutoff, flags);
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

int xnn_eeq_store_tiles(const double* pos, int64_t n_nodes, const double* cell, const double* rad,
                        double alpha, double cutoff, const xnn_eeq_tiles* tiles, int64_t* counts,
                        double* values, xnn_stream_t stream) {
  XNN_REQUIRE(n_nodes >= 0 && tiles != nullptr && tiles->n_tiles >= 0, "negative size or NULL tiles");
  if (n_nodes == 0 || tiles->n_tiles == 0) return XNN_OK;
  XNN_REQUIRE(pos && rad && tiles->tile_ij && tiles->mask && tiles->off, "NULL input or output");
  XNN_REQUIRE((values == nullptr) != (counts == nullptr), "either counts or values");
  XNN_REQUIRE(values == nullptr || tiles->base, "NULL tile bases");
  XNN_REQUIRE(n_nodes <= (int64_t(1) << 21) && tiles->n_tiles < (int64_t(1) << 31), "too many tiles");
  XNN_REQUIRE(cutoff > 0.0 && alpha >= 0.0, "cutoff must be positive, alpha non-negative");
  XNN_REQUIRE(cell != nullptr || alpha == 0.0, "a molecule takes alpha = 0");
  EeqCell C;
  XNN_REQUIRE(eeq_cell(cell, cutoff, C), "singular cell");
  XNN_REQUIRE(eeq_reach_ok(C, cutoff), "the real-space range spans more than %g cells",
              kMaxReach);
  const auto k = values != nullptr ? eeq_store_kernel<true> : eeq_store_kernel<false>;
  hipLaunchKernelGGL(k, dim3((unsigned)tiles->n_tiles), dim3(256), 0, as_hip(stream), pos, n_nodes,
                     C, rad, alpha, cutoff * cutoff, tiles->tile_ij, tiles->mask, tiles->off, counts,
                     tiles->base, values);
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

int xnn_eeq_store_apply_work_size(int64_t n_tiles, int32_t nrhs, size_t* bytes) {
  XNN_REQUIRE(n_tiles >= 0 && bytes != nullptr, "negative size or NULL output");
  XNN_REQUIRE(nrhs == 1 || nrhs == 2, "one or two right-hand sides (got %d)", (int)nrhs);
  *bytes = sizeof(double) * (size_t)(std::max<int64_t>(n_tiles, 1) * 2 * kStoreTile * nrhs);
  return XNN_OK;
}

int xnn_eeq_store_apply(const double* values, const xnn_eeq_tiles* tiles, int64_t n_nodes,
                        const double* v, int32_t nrhs, double* out, void* work, size_t work_bytes,
                        xnn_stream_t stream) {
  XNN_REQUIRE(n_nodes >= 0 && tiles != nullptr, "negative size or NULL tiles");
  size_t need = 0;
  const int rc = xnn_eeq_store_apply_work_size(tiles->n_tiles, nrhs, &need);
  if (rc != XNN_OK) return rc;
  if (n_nodes == 0) return XNN_OK;
  XNN_REQUIRE(values && v && out && work, "NULL input, output or workspace");
  XNN_REQUIRE(tiles->n_tiles > 0 && tiles->tile_ij && tiles->index && tiles->mask && tiles->off &&
                  tiles->base,
              "empty or NULL tile list");
  XNN_REQUIRE(n_nodes <= (int64_t(1) << 21) && tiles->n_tiles < (int64_t(1) << 31),
              "too many tiles");
  XNN_REQUIRE(work_bytes >= need, "workspace too small: %zu < %zu", work_bytes, need);
  hipStream_t s = as_hip(stream);
  const int64_t nt = (n_nodes + kStoreTile - 1) / kStoreTile;
  double* part = static_cast<double*>(work);
  const auto go = [&](auto apply, auto sum) {
    hipLaunchKernelGGL(apply, dim3((unsigned)tiles->n_tiles), dim3(256), 0, s, values,
                       tiles->tile_ij, tiles->mask, tiles->off, tiles->base, n_nodes, v, part);
    hipLaunchKernelGGL(sum, dim3((unsigned)nt), dim3(1024), 0, s, part, tiles->index, n_nodes, nt,
                       out);
  };
  if (nrhs == 1) go(eeq_tiles_apply_kernel<1>, eeq_tiles_sum_kernel<1>);
  else go(eeq_tiles_apply_kernel<2>, eeq_tiles_sum_kernel<2>);
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

int xnn_eeq_molecules(const double* pos, int64_t n_nodes, const int64_t* node_ptr,
                      const int32_t* ids, int64_t n_ids, int64_t max_atoms, const double* rad,
                      const double* diag, const double* x, const double* total, double* q,
                      int32_t* info, xnn_stream_t stream) {
  XNN_REQUIRE(n_nodes >= 0 && n_ids >= 0 && n_ids < (int64_t(1) << 31), "size out of range");
  if (n_nodes == 0 || n_ids == 0) return XNN_OK;
  XNN_REQUIRE(max_atoms >= 1 && max_atoms <= kMolMaxAtoms, "1 to %d atoms a molecule", kMolMaxAtoms);
  XNN_REQUIRE(pos && node_ptr && rad && diag && x && q && info, "NULL input or output");
  return launch_molecules<false>(pos, n_nodes, node_ptr, ids, n_ids, max_atoms, rad, diag, x, total,
                                 nullptr, q, nullptr, info, as_hip(stream));
}

int xnn_eeq_molecules_backward(const double* pos, int64_t n_nodes, const int64_t* node_ptr,
                               const int32_t* ids, int64_t n_ids, int64_t max_atoms,
                               const double* rad, const double* diag, const double* q,
                               const double* g_q, double* grad_pos, double* grad_x, int32_t* info,
                               xnn_stream_t stream) {
  XNN_REQUIRE(n_nodes >= 0 && n_ids >= 0 && n_ids < (int64_t(1) << 31), "size out of range");
  if (n_nodes == 0 || n_ids == 0) return XNN_OK;
  XNN_REQUIRE(max_atoms >= 1 && max_atoms <= kMolMaxAtoms, "1 to %d atoms a molecule", kMolMaxAtoms);
  XNN_REQUIRE(pos && node_ptr && rad && diag && q && g_q && grad_pos && grad_x && info,
              "NULL input or output");
  return launch_molecules<true>(pos, n_nodes, node_ptr, ids, n_ids, max_atoms, rad, diag, g_q,
                                nullptr, q, grad_x, grad_pos, info, as_hip(stream));
}

int xnn_eeq_cholesky_solve(const double* factor, int64_t n, const double* inv_blocks, double* x,
                           int32_t nrhs, double* work, xnn_stream_t stream) {
  XNN_REQUIRE(n >= 0, "negative size");
  XNN_REQUIRE(nrhs == 1 || nrhs == 2, "one or two right-hand sides (got %d)", (int)nrhs);
  if (n == 0) return XNN_OK;
  XNN_REQUIRE(factor && inv_blocks && x && work, "NULL factor, inverses, right-hand side or work");
  XNN_REQUIRE(n <= (int64_t(1) << 20), "at most 2^20 rows");
  return nrhs == 1 ? launch_trsv<1>(factor, n, inv_blocks, x, work, as_hip(stream))
                   : launch_trsv<2>(factor, n, inv_blocks, x, work, as_hip(stream));
}

int xnn_eeq_cholesky(double* matrix, int64_t n, double* inv_blocks, int* info,
                     xnn_stream_t stream) {
  XNN_REQUIRE(n >= 0 && n <= (int64_t(1) << 20), "0 to 2^20 rows");
  if (n == 0) return XNN_OK;
  XNN_REQUIRE(matrix && inv_blocks && info, "NULL matrix, inverses or info");
  hipStream_t s = as_hip(stream);
  for (int64_t k0 = 0; k0 < n; k0 += kCholBlock) {
    double* inv = inv_blocks + k0 * kCholBlock;
    const int64_t b = std::min<int64_t>(kCholBlock, n - k0), r0 = k0 + b;
    const int rc = launch_cholesky_block(matrix, n, k0, (int)b, inv, info, s);
    if (rc != XNN_OK) return rc;
    if (r0 == n) break;
    const int64_t rows = n - r0, m = (rows + kTrailTile - 1) / kTrailTile;
    hipLaunchKernelGGL(eeq_cholesky_panel_kernel,
                       dim3((unsigned)((rows + kPanelRows - 1) / kPanelRows)), dim3(256), 0, s, matrix,
                       n, k0, r0, inv);
    hipLaunchKernelGGL(eeq_cholesky_trail_kernel, dim3((unsigned)(m * (m + 1) / 2)), dim3(256), 0, s,
                       matrix, n, k0, r0);
  }
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

int xnn_eeq_cholesky_block(double* matrix, int64_t n, int64_t k0, int64_t b, double* inv,
                           int* info, xnn_stream_t stream) {
  XNN_REQUIRE(matrix && inv && info, "NULL matrix, inverse or info");
  XNN_REQUIRE(n > 0 && k0 >= 0 && b >= 1 && b <= kCholBlock && k0 + b <= n,
              "block [%lld, %lld) outside the matrix or wider than %d", (long long)k0,
              (long long)(k0 + b), kCholBlock);
  const int rc = launch_cholesky_block(matrix, n, k0, (int)b, inv, info, as_hip(stream));
  if (rc != XNN_OK) return rc;
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

}  // extern "C"
