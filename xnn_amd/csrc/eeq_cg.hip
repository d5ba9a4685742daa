// The vector work of the large EEQ regime's conjugate gradients (gfx950, float64), for one or
// two right-hand sides (common/models/eeq.py:325-360): everything of an iteration that is
// neither the real-space product nor a matrix product.
//
// The factorized reciprocal product A_rec v = Re[sum_k conj(P_k) (conj(B) (W S))_k], S =
// B^T (P v), is two library products with three launches around them:
//   spread: vp = [Re P v, Im P v] per atom, (rows, 2 K R);
//   fold:   the products' partial sums over row chunks -> S, times W, in the operand layout
//           [[gr, gi], [gi, -gr]] of the second product, (2 C, 2 K R);
//   gather: out_i += Re[conj(P_i) y_i] + diag_i v_i.
// An iteration's updates are these launches, most of which end in partial sums (one row per
// workgroup) that the next one adds up in every workgroup, in order:
//   dot:       p . Ap
//   step:      a = rz / p.Ap (0 for a column that is done); x += a p, r -= a Ap,
//              z = D^-1 r; r . r
//   project:   t = U^T z of the preconditioner's low-rank part (two launches)
//   direction: z -= D^-1 U t' (t' = core^-1 t, a library product); r . z
//   search:    b = rz' / rz; p = z + b p; rz = rz', done = |r| <= tolerance
// project and direction read U once each; as library products of two columns they compute
// tiles of 64 and 128. 24,000 atoms, 512 low-rank columns, two right-hand
// sides: project 30 + 6 us and direction 35 us (98 MB of U each, 3.3 and 2.8 TB/s), the other
// launches 5 to 12 us each; an iteration 0.95 ms, of which real space 0.36 and the reciprocal
// products 0.16, where some sixty tensor operations and four library products took 1.2 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "common.h"
#include "device.h"

namespace xnn {

constexpr int kCgThreads = 256;
constexpr int kCgBlocks = 256;        // workgroups, and rows of partial sums

static int cg_blocks(int64_t n) {
  return (int)std::min<int64_t>(kCgBlocks, (n + kCgThreads - 1) / kCgThreads);
}

static unsigned cg_grid(int64_t e) {
  return (unsigned)std::min<int64_t>(65536, (e + kCgThreads - 1) / kCgThreads);
}

// rows >= n of vp are zeros
__global__ __launch_bounds__(kCgThreads) void cg_spread_kernel(
    const double* __restrict__ pr, const double* __restrict__ pi, const double* __restrict__ v,
    int64_t n, int64_t rows, int K, int R, double* __restrict__ vp) {
  const int kr = K * R;
  for (int64_t e = (int64_t)blockIdx.x * kCgThreads + threadIdx.x; e < rows * kr;
       e += (int64_t)gridDim.x * kCgThreads) {
    const int64_t i = e / kr;
    const int q = (int)(e - i * kr), k = q / R, r = q - k * R;
    const double x = i < n ? v[i * R + r] : 0.0;
    const int64_t at = min(i, n - 1) * K + k;
    vp[i * 2 * kr + q] = pr[at] * x;
    vp[i * 2 * kr + kr + q] = pi[at] * x;
  }
}

// part (chunks, 2 C, 2 K R) -> out (2 C, 2 K R): four threads an element, a quarter of the
// chunks each
__global__ __launch_bounds__(kCgThreads) void cg_fold_kernel(const double* __restrict__ part,
                                                             int64_t chunks, int64_t C, int K,
                                                             int R, const double* __restrict__ W,
                                                             double* __restrict__ out) {
  constexpr int kPer = kCgThreads / kWave;
  __shared__ double sums[kPer][4][kWave];
  const int kr = K * R, lane = threadIdx.x & (kWave - 1), h = threadIdx.x / kWave;
  const int64_t e = (int64_t)blockIdx.x * kWave + lane, ec = min(e, C * kr - 1);
  const int64_t c = ec / kr, stride = 4 * C * kr;
  const int q = (int)(ec - c * kr);
  const double* lo = part + c * 2 * kr + q;
  const double* hi = lo + 2 * C * kr;
  double s[4] = {0.0, 0.0, 0.0, 0.0};                     // rr, ri, ir, ii
#pragma unroll 8
  for (int64_t m = h; m < chunks; m += kPer) {
    s[0] += lo[m * stride];
    s[1] += lo[m * stride + kr];
    s[2] += hi[m * stride];
    s[3] += hi[m * stride + kr];
  }
#pragma unroll
  for (int x = 0; x < 4; ++x) sums[h][x][lane] = s[x];
  __syncthreads();
  if (h != 0 || e >= C * kr) return;
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int g = 1; g < kPer; ++g) s[x] += sums[g][x][lane];
  const double w = W[c * K + q / R], gr = w * (s[0] - s[3]), gi = w * (s[1] + s[2]);
  out[c * 2 * kr + q] = gr;
  out[c * 2 * kr + kr + q] = gi;
  out[(C + c) * 2 * kr + q] = gi;
  out[(C + c) * 2 * kr + kr + q] = -gr;
}

// a wave per atom, lanes over the K phases
template <int R>
__global__ __launch_bounds__(kCgThreads) void cg_gather_kernel(
    const double* __restrict__ pr, const double* __restrict__ pi, const double* __restrict__ y,
    const double* __restrict__ diag, const double* __restrict__ v, int64_t n, int K,
    double* __restrict__ out) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t i = (int64_t)blockIdx.x * (kCgThreads / kWave) + threadIdx.x / kWave;
  if (i >= n) return;                                     // uniform in the wave
  const double* yi = y + i * 2 * K * R;
  double s[R];
#pragma unroll
  for (int r = 0; r < R; ++r) s[r] = 0.0;
  for (int k = lane; k < K; k += kWave) {
    const double c = pr[i * K + k], d = pi[i * K + k];
#pragma unroll
    for (int r = 0; r < R; ++r) s[r] += c * yi[k * R + r] + d * yi[(K + k) * R + r];
  }
#pragma unroll
  for (int m = kWave / 2; m > 0; m >>= 1)
#pragma unroll
    for (int r = 0; r < R; ++r) s[r] += __shfl_xor(s[r], m, kWave);
  if (lane == 0)
#pragma unroll
    for (int r = 0; r < R; ++r) out[i * R + r] += s[r] + diag[i] * v[i * R + r];
}

// the workgroup's sum of s (R columns) into part[blockIdx.x]; every thread calls it
template <int R, int THREADS = kCgThreads>
__device__ __forceinline__ void cg_block_sum(const double (&s)[R], double* __restrict__ part) {
  __shared__ double sh[THREADS / kWave][R];
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  double v[R];
#pragma unroll
  for (int r = 0; r < R; ++r) v[r] = s[r];
#pragma unroll
  for (int m = kWave / 2; m > 0; m >>= 1)
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] += __shfl_xor(v[r], m, kWave);
  if (lane == 0)
#pragma unroll
    for (int r = 0; r < R; ++r) sh[w][r] = v[r];
  __syncthreads();
  if (threadIdx.x == 0)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      double x = 0.0;
#pragma unroll
      for (int q = 0; q < THREADS / kWave; ++q) x += sh[q][r];
      part[blockIdx.x * R + r] = x;
    }
}

// the sum of the workgroups' partial sums, the same bits in every thread of every workgroup
template <int R>
__device__ __forceinline__ void cg_total(const double* __restrict__ part, int blocks, double (&out)[R]) {
  const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
  for (int r = 0; r < R; ++r) out[r] = 0.0;
  for (int b = lane; b < blocks; b += kWave)
#pragma unroll
    for (int r = 0; r < R; ++r) out[r] += part[b * R + r];
#pragma unroll
  for (int m = kWave / 2; m > 0; m >>= 1)
#pragma unroll
    for (int r = 0; r < R; ++r) out[r] += __shfl_xor(out[r], m, kWave);
}

template <int R>
__global__ __launch_bounds__(kCgThreads) void cg_dot_kernel(const double* __restrict__ a,
                                                            const double* __restrict__ b, int64_t n,
                                                            double* __restrict__ part) {
  double s[R];
#pragma unroll
  for (int r = 0; r < R; ++r) s[r] = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kCgThreads + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kCgThreads)
#pragma unroll
    for (int r = 0; r < R; ++r) s[r] = fma(a[i * R + r], b[i * R + r], s[r]);
  cg_block_sum<R>(s, part);
}

// state: rz (R), done (R) as 0 or 1
template <int R>
__global__ __launch_bounds__(kCgThreads) void cg_step_kernel(
    const double* __restrict__ pap, const double* __restrict__ state, const double* __restrict__ p,
    const double* __restrict__ ap, const double* __restrict__ inv_d, int64_t n,
    double* __restrict__ x, double* __restrict__ res, double* __restrict__ z,
    double* __restrict__ part) {
  double a[R], s[R];
  cg_total<R>(pap, gridDim.x, a);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    a[r] = state[R + r] != 0.0 ? 0.0 : state[r] / a[r];
    s[r] = 0.0;
  }
  for (int64_t i = (int64_t)blockIdx.x * kCgThreads + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kCgThreads)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int64_t e = i * R + r;
      x[e] = fma(a[r], p[e], x[e]);
      const double q = fma(-a[r], ap[e], res[e]);
      res[e] = q;
      z[e] = inv_d[i] * q;
      s[r] = fma(q, q, s[r]);
    }
  cg_block_sum<R>(s, part);
}

// part[block][l][r] = sum over the block's rows of U[i][l] z[i][r], a thread per column l
constexpr int kLowBlocks = 512;       // two workgroups a compute unit
constexpr int kLowRows = 32;          // rows staged at a time
constexpr int kLowLds = 2048;         // columns of U up to which t is in LDS (32 KB at most)

static int low_blocks(int64_t n) {
  return (int)std::min<int64_t>(kLowBlocks, (n + kLowRows - 1) / kLowRows);
}

template <int R>
__global__ __launch_bounds__(kCgThreads) void cg_project_kernel(const double* __restrict__ U,
                                                                const double* __restrict__ z,
                                                                int64_t n, int L, int64_t per,
                                                                double* __restrict__ part) {
  __shared__ double sz[kLowRows][R];
  const int64_t i0 = (int64_t)blockIdx.x * per, i1 = min(n, i0 + per);
  for (int l0 = 0; l0 < L; l0 += 2 * kCgThreads) {        // two columns a thread
    const int la = l0 + threadIdx.x, lb = la + kCgThreads;
    const int ca = min(la, L - 1), cb = min(lb, L - 1);
    double a[R], b[R];
#pragma unroll
    for (int r = 0; r < R; ++r) a[r] = b[r] = 0.0;
    for (int64_t base = i0; base < i1; base += kLowRows) {
      const int cnt = (int)min<int64_t>(kLowRows, i1 - base);
      __syncthreads();
      for (int e = threadIdx.x; e < kLowRows * R; e += kCgThreads)
        (&sz[0][0])[e] = e < cnt * R ? z[base * R + e] : 0.0;
      __syncthreads();
#pragma unroll 8
      for (int j = 0; j < cnt; ++j) {
        const double ua = U[(base + j) * L + ca], ub = U[(base + j) * L + cb];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          a[r] = fma(ua, sz[j][r], a[r]);
          b[r] = fma(ub, sz[j][r], b[r]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (la < L) part[((int64_t)blockIdx.x * L + la) * R + r] = a[r];
      if (lb < L) part[((int64_t)blockIdx.x * L + lb) * R + r] = b[r];
    }
  }
}

// out[e] = sum of part[block][e] over the blocks: sixteen threads an element
__global__ __launch_bounds__(kCgThreads) void cg_project_sum_kernel(const double* __restrict__ part,
                                                                    int blocks, int m,
                                                                    double* __restrict__ out) {
  __shared__ double s[16][17];
  const int x = threadIdx.x % 16, y = threadIdx.x / 16, e = blockIdx.x * 16 + x;
  double v = 0.0;
  if (e < m) {
#pragma unroll 8
    for (int b = y; b < blocks; b += 16) v += part[(int64_t)b * m + e];
  }
  s[y][x] = v;
  __syncthreads();
  if (y == 0 && e < m) {
    double r = 0.0;
#pragma unroll
    for (int q = 0; q < 16; ++q) r += s[q][x];
    out[e] = r;
  }
}

// U NULL: no low-rank part. A wave per row, lanes over the columns of U, t in LDS (LDS) or from
// L2
constexpr int kDirThreads = 1024;

template <int R, bool LDS>
__global__ __launch_bounds__(kDirThreads) void cg_direction_kernel(
    const double* __restrict__ U, const double* __restrict__ t, int L,
    const double* __restrict__ inv_d, const double* __restrict__ res, int64_t n,
    double* __restrict__ z, double* __restrict__ part) {
  extern __shared__ double st[];                          // [r][l]
  double s[R];
#pragma unroll
  for (int r = 0; r < R; ++r) s[r] = 0.0;
  if (U == nullptr) {
    for (int64_t i = (int64_t)blockIdx.x * kDirThreads + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kDirThreads)
#pragma unroll
      for (int r = 0; r < R; ++r) s[r] = fma(res[i * R + r], z[i * R + r], s[r]);
  } else {
    if constexpr (LDS) {
      for (int e = threadIdx.x; e < L * R; e += kDirThreads) st[(e % R) * L + e / R] = t[e];
      __syncthreads();
    }
    const int lane = threadIdx.x & (kWave - 1);
    constexpr int kWaves = kDirThreads / kWave;
    for (int64_t i = (int64_t)blockIdx.x * kWaves + threadIdx.x / kWave; i < n;
         i += (int64_t)gridDim.x * kWaves) {
      double u[R];
#pragma unroll
      for (int r = 0; r < R; ++r) u[r] = 0.0;
#pragma unroll 8
      for (int l = lane; l < L; l += kWave) {
        const double x = U[i * L + l];
#pragma unroll
        for (int r = 0; r < R; ++r) u[r] = fma(x, LDS ? st[r * L + l] : t[l * R + r], u[r]);
      }
#pragma unroll
      for (int m = kWave / 2; m > 0; m >>= 1)
#pragma unroll
        for (int r = 0; r < R; ++r) u[r] += __shfl_xor(u[r], m, kWave);
      if (lane == 0)
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const double q = fma(-inv_d[i], u[r], z[i * R + r]);
          z[i * R + r] = q;
          s[r] = fma(res[i * R + r], q, s[r]);
        }
    }
  }
  cg_block_sum<R, kDirThreads>(s, part);
}

// first: p = z
template <int R>
__global__ __launch_bounds__(kCgThreads) void cg_search_kernel(
    const double* __restrict__ rz, const double* __restrict__ rr, const double* __restrict__ tol,
    const double* __restrict__ old, bool first, const double* __restrict__ z, int64_t n,
    double* __restrict__ p, double* __restrict__ state) {
  double b[R], sum[R], norm[R];
  cg_total<R>(rz, gridDim.x, sum);
  cg_total<R>(rr, gridDim.x, norm);
#pragma unroll
  for (int r = 0; r < R; ++r) b[r] = first || old[R + r] != 0.0 ? 0.0 : sum[r] / old[r];
  for (int64_t i = (int64_t)blockIdx.x * kCgThreads + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kCgThreads)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int64_t e = i * R + r;
      p[e] = first ? z[e] : fma(b[r], p[e], z[e]);
    }
  if (blockIdx.x == 0 && threadIdx.x == 0)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      state[r] = sum[r];
      state[R + r] = sqrt(norm[r]) <= tol[r] ? 1.0 : 0.0;
    }
}

}  // namespace xnn

using namespace xnn;

#define XNN_CG(K, N, ...)                                                                          \
  do {                                                                                             \
    if (nrhs == 1)                                                                                 \
      hipLaunchKernelGGL(K<1>, dim3((unsigned)cg_blocks(N)), dim3(kCgThreads), 0, s, __VA_ARGS__); \
    else                                                                                           \
      hipLaunchKernelGGL(K<2>, dim3((unsigned)cg_blocks(N)), dim3(kCgThreads), 0, s, __VA_ARGS__); \
    XNN_LAUNCH_CHECK();                                                                            \
  } while (0)

extern "C" {

int xnn_eeq_cg_spread(const double* pr, const double* pi, const double* v, int64_t n_nodes,
                      int64_t n_rows, int32_t n_phases, int32_t nrhs, double* vp,
                      xnn_stream_t stream) {
  XNN_REQUIRE(n_nodes >= 1 && n_rows >= n_nodes && n_phases >= 1, "size out of range");
  XNN_REQUIRE(nrhs == 1 || nrhs == 2, "one or two right-hand sides (got %d)", (int)nrhs);
  XNN_REQUIRE(pr && pi && v && vp, "NULL input or output");
  hipLaunchKernelGGL(cg_spread_kernel, dim3(cg_grid(n_rows * n_phases * nrhs)), dim3(kCgThreads), 0,
                     as_hip(stream), pr, pi, v, n_nodes, n_rows, (int)n_phases, (int)nrhs, vp);
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

int xnn_eeq_cg_fold(const double* part, int64_t chunks, int64_t n_columns, int32_t n_phases,
                    int32_t nrhs, const double* weights, double* out, xnn_stream_t stream) {
  XNN_REQUIRE(chunks >= 1 && n_columns >= 1 && n_phases >= 1, "size out of range");
  XNN_REQUIRE(nrhs == 1 || nrhs == 2, "one or two right-hand sides (got %d)", (int)nrhs);
  XNN_REQUIRE(part && weights && out, "NULL input or output");
  const int64_t blocks = (n_columns * n_phases * nrhs + kWave - 1) / kWave;
  XNN_REQUIRE(blocks <= 0x7fffffff, "size out of range");
  hipLaunchKernelGGL(cg_fold_kernel, dim3((unsigned)blocks), dim3(kCgThreads), 0, as_hip(stream), part,
                     chunks, n_columns, (int)n_phases, (int)nrhs, weights, out);
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

int xnn_eeq_cg_gather(const double* pr, const double* pi, const double* y, const double* diag,
                      const double* v, int64_t n_nodes, int32_t n_phases, int32_t nrhs, double* out,
                      xnn_stream_t stream) {
  XNN_REQUIRE(n_nodes >= 1 && n_phases >= 1, "size out of range");
  XNN_REQUIRE(nrhs == 1 || nrhs == 2, "one or two right-hand sides (got %d)", (int)nrhs);
  XNN_REQUIRE(pr && pi && y && diag && v && out, "NULL input or output");
  constexpr int kWaves = kCgThreads / kWave;
  XNN_REQUIRE(n_nodes <= (int64_t)kWaves * 0x7fffffff, "too many atoms");
  const dim3 grid((unsigned)((n_nodes + kWaves - 1) / kWaves));
  if (nrhs == 1)
    hipLaunchKernelGGL(cg_gather_kernel<1>, grid, dim3(kCgThreads), 0, as_hip(stream), pr, pi, y, diag, v,
                       n_nodes, (int)n_phases, out);
  else
    hipLaunchKernelGGL(cg_gather_kernel<2>, grid, dim3(kCgThreads), 0, as_hip(stream), pr, pi, y, diag, v,
                       n_nodes, (int)n_phases, out);
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

int xnn_eeq_cg_step(const double* p, const double* ap, const double* inv_d, const double* state,
                    int64_t n_nodes, int32_t nrhs, double* x, double* res, double* z, double* sums,
                    xnn_stream_t stream) {
  XNN_REQUIRE(n_nodes >= 1, "size out of range");
  XNN_REQUIRE(nrhs == 1 || nrhs == 2, "one or two right-hand sides (got %d)", (int)nrhs);
  XNN_REQUIRE(p && ap && inv_d && state && x && res && z && sums, "NULL input or output");
  hipStream_t s = as_hip(stream);
  XNN_CG(cg_dot_kernel, n_nodes, p, ap, n_nodes, sums);
  XNN_CG(cg_step_kernel, n_nodes, sums, state, p, ap, inv_d, n_nodes, x, res, z, sums + nrhs * kCgBlocks);
  return XNN_OK;
}

int xnn_eeq_cg_project_work_size(int64_t n_nodes, int32_t n_low, int32_t nrhs, size_t* bytes) {
  XNN_REQUIRE(bytes != nullptr, "NULL size");
  XNN_REQUIRE(n_nodes >= 1 && n_low >= 1 && nrhs >= 1, "size out of range");
  *bytes = sizeof(double) * (size_t)low_blocks(n_nodes) * n_low * nrhs;
  return XNN_OK;
}

int xnn_eeq_cg_project(const double* U, const double* z, int64_t n_nodes, int32_t n_low,
                       int32_t nrhs, double* t, void* work, size_t work_bytes,
                       xnn_stream_t stream) {
  XNN_REQUIRE(n_nodes >= 1 && n_low >= 1 && n_low < (1 << 29), "size out of range");
  XNN_REQUIRE(nrhs == 1 || nrhs == 2, "one or two right-hand sides (got %d)", (int)nrhs);
  XNN_REQUIRE(U && z && t && work, "NULL input, output or work");
  const int want = low_blocks(n_nodes), m = n_low * nrhs;
  XNN_REQUIRE(work_bytes >= sizeof(double) * (size_t)want * m, "work too small");
  const int64_t per = (n_nodes + want - 1) / want;
  const int blocks = (int)((n_nodes + per - 1) / per);
  hipStream_t s = as_hip(stream);
  double* part = static_cast<double*>(work);
  if (nrhs == 1)
    hipLaunchKernelGGL(cg_project_kernel<1>, dim3(blocks), dim3(kCgThreads), 0, s, U, z, n_nodes,
                       (int)n_low, per, part);
  else
    hipLaunchKernelGGL(cg_project_kernel<2>, dim3(blocks), dim3(kCgThreads), 0, s, U, z, n_nodes,
                       (int)n_low, per, part);
  hipLaunchKernelGGL(cg_project_sum_kernel, dim3((m + 15) / 16), dim3(kCgThreads), 0, s, part, blocks, m,
                     t);
  XNN_LAUNCH_CHECK();
  return XNN_OK;
}

int xnn_eeq_cg_search(const double* U, const double* t, int32_t n_low, const double* inv_d,
                      const double* res, const double* tol, const double* state, int32_t first,
                      int64_t n_nodes, int32_t nrhs, double* z, double* p, double* new_state,
                      double* sums, xnn_stream_t stream) {
  XNN_REQUIRE(n_nodes >= 1, "size out of range");
  XNN_REQUIRE(nrhs == 1 || nrhs == 2, "one or two right-hand sides (got %d)", (int)nrhs);
  XNN_REQUIRE(inv_d && res && tol && (first || state) && z && p && new_state && sums,
              "NULL input or output");
  XNN_REQUIRE(U == nullptr || (t && n_low >= 1 && n_low < (1 << 29)), "NULL t or size out of range");
  XNN_REQUIRE(state != new_state, "the state is read while the new one is written");
  hipStream_t s = as_hip(stream);
  if (first) XNN_CG(cg_dot_kernel, n_nodes, res, res, n_nodes, sums + nrhs * kCgBlocks);
  const bool low_lds = U != nullptr && n_low <= kLowLds;
  const size_t lds = low_lds ? sizeof(double) * (size_t)n_low * nrhs : 0;
  const auto direction =
      nrhs == 1 ? (low_lds ? cg_direction_kernel<1, true> : cg_direction_kernel<1, false>)
                : (low_lds ? cg_direction_kernel<2, true> : cg_direction_kernel<2, false>);
  hipLaunchKernelGGL(direction, dim3((unsigned)cg_blocks(n_nodes)), dim3(kDirThreads), lds, s, U, t,
                     (int)n_low, inv_d, res, n_nodes, z, sums);
  XNN_CG(cg_search_kernel, n_nodes, sums, sums + nrhs * kCgBlocks, tol, state, first != 0, z, n_nodes, p,
         new_state);
  return XNN_OK;
}

}  // extern "C"
