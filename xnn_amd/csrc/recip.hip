// The reciprocal part of the Ewald product of the large EEQ regime and its derivatives
// (gfx950, float64): out = C diag(w) C^T v + S diag(w) S^T v with C, S = cos, sin(pos G^T)
// (common/models/eeq.py:170-397). The (N, M) phases are never stored: a sum over the atoms
// with a thread per vector gives the structure factors S_k = sum_i v_i (cos, sin)(G_k . r_i),
// a sum over the vectors with a thread per atom the result. The backward for the output's
// gradient u takes one pass of each kind: with the factors T_k of u,
//   dL/dr_i = sum_k w_k G_k [cos (u_i Ss + v_i Ts) - sin (u_i Sc + v_i Tc)],
//   dL/dv_i = sum_k w_k [Tc cos + Ts sin],    dL/dw_k = Sc Tc + Ss Ts,
//   dL/dG_k = w_k [Ss sum_i cos u_i r_i + Ts sum_i cos v_i r_i
//                  - Sc sum_i sin u_i r_i - Tc sum_i sin v_i r_i],
// the four moments of the last being accumulated with T. Sums are split over workgroups and
// added in a fixed order: the same bits every time.
// Bound by the float64 sine and cosine, 26 to 34 us for each of the four passes over 5,000
// atoms (8 million phases each); the stored phases' products, their matrix-vector sums and the
// phases' gradient took 1,600 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "common.h"
#include "device.h"

namespace xnn {

constexpr int kRecipTile = 256;      // threads, and terms staged at a time
constexpr int kRecipBlocks = 2048;   // target workgroups a launch: 8 per CU
constexpr int kRecipMinTerms = 64;   // fewer terms a workgroup and the partial sums dominate

static int64_t recip_splits(int64_t rows, int64_t terms) {
  const int64_t tiles = (rows + kRecipTile - 1) / kRecipTile;
  return std::max<int64_t>(1, std::min((terms + kRecipMinTerms - 1) / kRecipMinTerms,
                                       (kRecipBlocks + tiles - 1) / tiles));
}

// part[split][q][k], q: Q = 2: sums of v (cos, sin); Q = 14: sums of u (cos, sin), then
// (cos u r, cos v r, sin u r, sin v r), three components each
template <int Q>
__global__ __launch_bounds__(kRecipTile) void recip_factors_kernel(
    const double* __restrict__ pos, int64_t n, const double* __restrict__ g, int64_t m,
    const double* __restrict__ v, const double* __restrict__ u, int64_t chunk,
    double* __restrict__ part) {
  __shared__ double sp[3][kRecipTile], sv[kRecipTile], su[Q > 2 ? kRecipTile : 1];
  const int t = threadIdx.x;
  const int64_t k = (int64_t)blockIdx.x * kRecipTile + t, kc = min(k, m - 1);
  const int64_t i0 = (int64_t)blockIdx.y * chunk, i1 = min(n, i0 + chunk);
  const double g0 = g[3 * kc], g1 = g[3 * kc + 1], g2 = g[3 * kc + 2];
  double acc[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) acc[q] = 0.0;
  for (int64_t b = i0; b < i1; b += kRecipTile) {
    const int cnt = (int)min<int64_t>(kRecipTile, i1 - b);
    __syncthreads();
    if (t < cnt) {
#pragma unroll
      for (int c = 0; c < 3; ++c) sp[c][t] = pos[3 * (b + t) + c];
      sv[t] = v[b + t];
      if (Q > 2) su[t] = u[b + t];
    }
    __syncthreads();
    for (int j = 0; j < cnt; ++j) {
      const double r[3] = {sp[0][j], sp[1][j], sp[2][j]};
      double s, c;
      sincos(fma(g2, r[2], fma(g1, r[1], g0 * r[0])), &s, &c);
      const double lead = Q > 2 ? su[j] : sv[j];
      acc[0] = fma(lead, c, acc[0]);
      acc[1] = fma(lead, s, acc[1]);
      if constexpr (Q > 2) {
        const double cu = c * su[j], cv = c * sv[j], du = s * su[j], dv = s * sv[j];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          acc[2 + a] = fma(cu, r[a], acc[2 + a]);
          acc[5 + a] = fma(cv, r[a], acc[5 + a]);
          acc[8 + a] = fma(du, r[a], acc[8 + a]);
          acc[11 + a] = fma(dv, r[a], acc[11 + a]);
        }
      }
    }
  }
  if (k < m) {
#pragma unroll
    for (int q = 0; q < Q; ++q) part[((int64_t)blockIdx.y * Q + q) * m + k] = acc[q];
  }
}

// part[split][q][i]: BWD false: q = 0 the product; true: q = 0..2 the gradient of r_i, 3 of v_i
template <bool BWD>
__global__ __launch_bounds__(kRecipTile) void recip_atoms_kernel(
    const double* __restrict__ pos, int64_t n, const double* __restrict__ g,
    const double* __restrict__ w, int64_t m, const double* __restrict__ fs,
    const double* __restrict__ ft, const double* __restrict__ v, const double* __restrict__ u,
    int64_t chunk, double* __restrict__ part) {
  constexpr int Q = BWD ? 4 : 1;
  __shared__ double sg[3][kRecipTile], sa[2][kRecipTile], st[BWD ? 2 : 1][BWD ? kRecipTile : 1];
  const int t = threadIdx.x;
  const int64_t i = (int64_t)blockIdx.x * kRecipTile + t, ic = min(i, n - 1);
  const int64_t k0 = (int64_t)blockIdx.y * chunk, k1 = min(m, k0 + chunk);
  const double x = pos[3 * ic], y = pos[3 * ic + 1], z = pos[3 * ic + 2];
  const double vi = BWD ? v[ic] : 0.0, ui = BWD ? u[ic] : 0.0;
  double acc[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) acc[q] = 0.0;
  for (int64_t b = k0; b < k1; b += kRecipTile) {
    const int cnt = (int)min<int64_t>(kRecipTile, k1 - b);
    __syncthreads();
    if (t < cnt) {
#pragma unroll
      for (int c = 0; c < 3; ++c) sg[c][t] = g[3 * (b + t) + c];
      const double wk = w[b + t];
      sa[0][t] = wk * fs[b + t];
      sa[1][t] = wk * fs[m + b + t];
      if constexpr (BWD) {
        st[0][t] = wk * ft[b + t];
        st[1][t] = wk * ft[m + b + t];
      }
    }
    __syncthreads();
    for (int j = 0; j < cnt; ++j) {
      double s, c;
      sincos(fma(sg[2][j], z, fma(sg[1][j], y, sg[0][j] * x)), &s, &c);
      if constexpr (BWD) {
        const double f = c * fma(ui, sa[1][j], vi * st[1][j]) - s * fma(ui, sa[0][j], vi * st[0][j]);
#pragma unroll
        for (int a = 0; a < 3; ++a) acc[a] = fma(f, sg[a][j], acc[a]);
        acc[3] = fma(st[0][j], c, fma(st[1][j], s, acc[3]));
      } else {
        acc[0] = fma(sa[0][j], c, fma(sa[1][j], s, acc[0]));
      }
    }
  }
  if (i < n) {
#pragma unroll
    for (int q = 0; q < Q; ++q) part[((int64_t)blockIdx.y * Q + q) * n + i] = acc[q];
  }
}

// out[e] = sum over the splits of part[split][e], e < rows, in split order
__global__ __launch_bounds__(kRecipTile) void recip_sum_kernel(const double* __restrict__ part,
                                                               int64_t splits, int64_t rows,
                                                               double* __restrict__ out) {
  const int64_t e = (int64_t)blockIdx.x * kRecipTile + threadIdx.x;
  if (e >= rows) return;
  double s = 0.0;
#pragma unroll 8
  for (int64_t q = 0; q < splits; ++q) s += part[q * rows + e];
  out[e] = s;
}

// the atoms' sums, component-major, to the outputs
__global__ __launch_bounds__(kRecipTile) void recip_atom_grads_kernel(
    const double* __restrict__ part, int64_t splits, int64_t n, double* __restrict__ grad_pos,
    double* __restrict__ grad_v) {
  const int64_t e = (int64_t)blockIdx.x * kRecipTile + threadIdx.x;
  if (e >= 4 * n) return;
  double s = 0.0;
#pragma unroll 8
  for (int64_t q = 0; q < splits; ++q) s += part[q * 4 * n + e];
  const int64_t a = e / n, i = e % n;
  if (a < 3)
    grad_pos[3 * i + a] = s;
  else if (grad_v != nullptr)
    grad_v[i] = s;
}

__global__ __launch_bounds__(kRecipTile) void recip_vector_grads_kernel(
    const double* __restrict__ w, int64_t m, const double* __restrict__ fs,
    const double* __restrict__ ft, double* __restrict__ grad_g, double* __restrict__ grad_w) {
  const int64_t k = (int64_t)blockIdx.x * kRecipTile + threadIdx.x;
  if (k >= m) return;
  const double sc = fs[k], ss = fs[m + k], tc = ft[k], ts = ft[m + k];
#pragma unroll
  for (int a = 0; a < 3; ++a)
    grad_g[3 * k + a] = w[k] * (ss * ft[(2 + a) * m + k] + ts * ft[(5 + a) * m + k] -
                                sc * ft[(8 + a) * m + k] - tc * ft[(11 + a) * m + k]);
  grad_w[k] = fma(sc, tc, ss * ts);
}

static unsigned recip_tiles(int64_t rows) { return (unsigned)((rows + kRecipTile - 1) / kRecipTile); }

static int64_t recip_work(int64_t n, int64_t m, int backward) {
  const int64_t fs = recip_splits(m, n), as = recip_splits(n, m);
  return backward ? 14 * m * (fs + 1) + 4 * n * as : std::max(2 * m * fs, n * as);
}

}  // namespace xnn

using namespace xnn;

extern "C" {

int xnn_eeq_recip_work_size(int64_t n_nodes, int64_t n_vectors, int32_t backward, size_t* bytes) {
  XNN_REQUIRE(bytes != nullptr, "NULL size");
  XNN_REQUIRE(n_nodes >= 0 && n_vectors >= 0, "negative size");
  *bytes = n_nodes == 0 || n_vectors == 0
               ? 0 : sizeof(double) * (size_t)recip_work(n_nodes, n_vectors, backward);
  return XNN_OK;
}

int xnn_eeq_recip(const double* pos, int64_t n_nodes, const double* g, const double* w,
                  int64_t n_vectors, const double* v, double* factors, double* out, void* work,
                  size_t work_bytes, xnn_stream_t stream) {
  const int64_t n = n_nodes, m = n_vectors;
  XNN_REQUIRE(n >= 0 && m >= 0 && n < (int64_t(1) << 31) && m < (int64_t(1) << 31), "size out of range");
  if (n == 0 || m == 0) return XNN_OK;
  XNN_REQUIRE(pos && g && w && v && factors && out && work, "NULL input, output or work");
  XNN_REQUIRE(work_bytes >= sizeof(double) * (size_t)recip_work(n, m, 0), "work too small");
  hipStream_t s = as_hip(stream);
  double* part = static_cast<double*>(work);
  const int64_t fs = recip_splits(m, n), as = recip_splits(n, m);
  hipLaunchKernelGGL(recip_factors_kernel<2>, dim3(recip_tiles(m), (unsigned)fs), dim3(kRecipTile), 0,
                     s, pos, n, g, m, v, nullptr, (n + fs - 1) / fs, part);
  hipLaunchKernelGGL(recip_sum_kernel, dim3(recip_tiles(2 * m)), dim3(kRecipTile), 0, s, part, fs,
                     2 * m, factors);
  hipLaunchKernelGGL(recip_atoms_kernel<false>, dim3(recip_tiles(n), (unsigned)as), dim3(kRecipTile), 0,
                     s, pos, n, g, w, m, factors, nullptr, nullptr, nullptr, (m + as - 1) / as, part);
  hipLaunchKernelGGL(recip_sum_kernel, dim3(recip_tiles(n)), dim3(kRecipTile), 0, s, part, as, n, out);
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

int xnn_eeq_recip_backward(const double* pos, int64_t n_nodes, const double* g, const double* w,
                           int64_t n_vectors, const double* v, const double* factors,
                           const double* u, double* grad_pos, double* grad_g, double* grad_w,
                           double* grad_v, void* work, size_t work_bytes, xnn_stream_t stream) {
  const int64_t n = n_nodes, m = n_vectors;
  XNN_REQUIRE(n >= 0 && m >= 0 && n < (int64_t(1) << 31) && m < (int64_t(1) << 31), "size out of range");
  if (n == 0 || m == 0) return XNN_OK;
  XNN_REQUIRE(pos && g && w && v && factors && u && grad_pos && work, "NULL input, output or work");
  XNN_REQUIRE((grad_g == nullptr) == (grad_w == nullptr), "the vectors' and weights' gradients together");
  XNN_REQUIRE(work_bytes >= sizeof(double) * (size_t)recip_work(n, m, 1), "work too small");
  hipStream_t s = as_hip(stream);
  const int64_t fs = recip_splits(m, n), as = recip_splits(n, m), per = (n + fs - 1) / fs;
  double* ft = static_cast<double*>(work);                // 14 m, then the partial sums
  double* fpart = ft + 14 * m;
  double* apart = fpart + 14 * m * fs;
  const dim3 grid(recip_tiles(m), (unsigned)fs);
  const int64_t rows = grad_g != nullptr ? 14 * m : 2 * m;
  if (grad_g != nullptr)
    hipLaunchKernelGGL(recip_factors_kernel<14>, grid, dim3(kRecipTile), 0, s, pos, n, g, m, v, u, per,
                       fpart);
  else
    hipLaunchKernelGGL(recip_factors_kernel<2>, grid, dim3(kRecipTile), 0, s, pos, n, g, m, u, nullptr,
                       per, fpart);
  hipLaunchKernelGGL(recip_sum_kernel, dim3(recip_tiles(rows)), dim3(kRecipTile), 0, s, fpart, fs, rows,
                     ft);
  hipLaunchKernelGGL(recip_atoms_kernel<true>, dim3(recip_tiles(n), (unsigned)as), dim3(kRecipTile), 0,
                     s, pos, n, g, w, m, factors, ft, v, u, (m + as - 1) / as, apart);
  hipLaunchKernelGGL(recip_atom_grads_kernel, dim3(recip_tiles(4 * n)), dim3(kRecipTile), 0, s, apart,
                     as, n, grad_pos, grad_v);
  if (grad_g != nullptr)
    hipLaunchKernelGGL(recip_vector_grads_kernel, dim3(recip_tiles(m)), dim3(kRecipTile), 0, s, w, m,
                       factors, ft, grad_g, grad_w);
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

}  // extern "C"
