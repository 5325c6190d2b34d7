// Kernels of the full-update bond step (acetn/evolution/full_update.py,
// als_solver.py, tensor_update.py): tiny dense linear algebra that runs in
// one workgroup per problem (latency-bound; the matrices are 6x6 .. 1728x12),
// the persistent ALS solver, and a strided permute-copy.
#include "internal.h"
#include "fu_internal.h"
#include "lanes.h"

#include <algorithm>
#include <type_traits>
#include <cmath>

namespace acetn {
namespace {

// ---------------------------------------------------------------------------
// permute-copy: out (contiguous, dims od[0..n-1]) = scale * in[sum_i idx_i * is[i]]
// ---------------------------------------------------------------------------
__global__ void permute_kernel(const double* __restrict__ in, double* __restrict__ out,
                               PermDesc p, double scale) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < p.total;
       e += (int64_t)gridDim.x * blockDim.x) {
    int64_t r = e, off = 0;
    for (int i = p.n - 1; i >= 0; --i) {
      const int64_t x = r % p.od[i];
      r /= p.od[i];
      off += x * p.is[i];
    }
    out[e] = scale * in[off];
  }
}

// ---------------------------------------------------------------------------
// Householder QR of a dense row-major m x n matrix (n <= kQrMaxN), one
// workgroup.  Conventions of LAPACK dgeqrf/dorgqr (and so of numpy.linalg.qr):
// beta = -sign(alpha) * ||x||, R[j][j] = beta, thin Q formed by backward
// accumulation.  W (m x n) is scratch and receives the reflectors.
// ---------------------------------------------------------------------------
constexpr int QR_NT = 256;

__device__ double block_sum(double v, double* red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += red[w];
  return t;
}

__global__ __launch_bounds__(QR_NT) void householder_qr_kernel(const double* __restrict__ A,
                                                               int m, int n,
                                                               double* __restrict__ W,
                                                               double* __restrict__ Q,
                                                               double* __restrict__ R) {
  __shared__ double red[QR_NT / 64];
  __shared__ double part[QR_NT / 64][kQrMaxN];
  __shared__ double tau[kQrMaxN], wv[kQrMaxN];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int64_t e = tid; e < (int64_t)m * n; e += QR_NT) W[e] = A[e];
  __syncthreads();
  const int kmax = min(m, n);
  for (int j = 0; j < kmax; ++j) {
    double xs = 0.0;
    for (int i = j + 1 + tid; i < m; i += QR_NT) xs += W[(int64_t)i * n + j] * W[(int64_t)i * n + j];
    const double xnorm2 = block_sum(xs, red);
    const double alpha = W[(int64_t)j * n + j];
    double beta = alpha, t = 0.0, scal = 0.0;
    if (xnorm2 > 0.0) {
      beta = -copysign(sqrt(alpha * alpha + xnorm2), alpha);
      t = (beta - alpha) / beta;
      scal = 1.0 / (alpha - beta);
    }
    __syncthreads();
    if (tid == 0) { tau[j] = t; W[(int64_t)j * n + j] = beta; }
    for (int i = j + 1 + tid; i < m; i += QR_NT) W[(int64_t)i * n + j] *= scal;
    __syncthreads();
    if (t != 0.0 && j + 1 < n) {
      // w_c = v^T W[:, c] for c > j  (v_j = 1)
      double acc[kQrMaxN];
#pragma unroll
      for (int c = 0; c < kQrMaxN; ++c) acc[c] = 0.0;
      for (int i = j + tid; i < m; i += QR_NT) {
        const double vi = (i == j) ? 1.0 : W[(int64_t)i * n + j];
#pragma unroll
        for (int c = 0; c < kQrMaxN; ++c)
          if (c > j && c < n) acc[c] += vi * W[(int64_t)i * n + c];
      }
#pragma unroll
      for (int c = 0; c < kQrMaxN; ++c) {
        double v = acc[c];
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
        if (lane == 0) part[wave][c] = v;
      }
      __syncthreads();
      if (tid < n) {
        double s = 0.0;
        for (int w = 0; w < QR_NT / 64; ++w) s += part[w][tid];
        wv[tid] = s;
      }
      __syncthreads();
      for (int i = j + tid; i < m; i += QR_NT) {
        const double vi = (i == j) ? 1.0 : W[(int64_t)i * n + j];
        for (int c = j + 1; c < n; ++c) W[(int64_t)i * n + c] -= t * vi * wv[c];
      }
      __syncthreads();
    }
  }
  // R (n x n, upper; rows beyond kmax are zero)
  for (int e = tid; e < n * n; e += QR_NT) {
    const int r = e / n, c = e % n;
    R[e] = (r <= c && r < kmax) ? W[(int64_t)r * n + c] : 0.0;
  }
  if (Q == nullptr) return;
  // thin Q = H_0 ... H_{kmax-1} I[:, :kmax]  (m x kmax, leading dimension n)
  for (int64_t e = tid; e < (int64_t)m * n; e += QR_NT) {
    const int r = (int)(e / n), c = (int)(e % n);
    Q[e] = (r == c) ? 1.0 : 0.0;
  }
  __syncthreads();
  for (int j = kmax - 1; j >= 0; --j) {
    const double t = tau[j];
    if (t == 0.0) continue;
    double acc[kQrMaxN];
#pragma unroll
    for (int c = 0; c < kQrMaxN; ++c) acc[c] = 0.0;
    for (int i = j + tid; i < m; i += QR_NT) {
      const double vi = (i == j) ? 1.0 : W[(int64_t)i * n + j];
#pragma unroll
      for (int c = 0; c < kQrMaxN; ++c)
        if (c >= j && c < kmax) acc[c] += vi * Q[(int64_t)i * n + c];
    }
#pragma unroll
    for (int c = 0; c < kQrMaxN; ++c) {
      double v = acc[c];
      for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
      if (lane == 0) part[wave][c] = v;
    }
    __syncthreads();
    if (tid < n) {
      double s = 0.0;
      for (int w = 0; w < QR_NT / 64; ++w) s += part[w][tid];
      wv[tid] = s;
    }
    __syncthreads();
    for (int i = j + tid; i < m; i += QR_NT) {
      const double vi = (i == j) ? 1.0 : W[(int64_t)i * n + j];
      for (int c = j; c < kmax; ++c) Q[(int64_t)i * n + c] -= t * vi * wv[c];
    }
    __syncthreads();
  }
}

// The same factorisation with the whole matrix in registers, up to 64 NWV R
// rows and NC columns, one workgroup per problem (one or two): row i is in
// thread i mod 64 NWV.  A column costs one exchange: the products of column j
// with itself and with all later ones are summed together (v^T W[:, c] =
// W[j][c] + (sum_{i > j} W[i][j] W[i][c]) / (alpha - beta)), where the kernel
// above makes three passes over memory and three block sums.  The input is
// read through its permutation (rows of up to three digits, columns of two).
// Latency-bound: 216 x 12 (D=6, d=2) 26 us the pair against 246 us each.
template <int NC, int R, int NWV>
__global__ __launch_bounds__(64 * NWV) void qr_reg_kernel(QrProblem p0, QrProblem p1, int m, int n) {
  constexpr int NT = 64 * NWV;
  __shared__ double part[2][NWV][NC], rowj[2][NC];
  const QrProblem& p = blockIdx.x ? p1 : p0;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kmax = min(m, n);
  double w[R][NC];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = min(tid + NT * r, m - 1);
    const int64_t ro = (int64_t)(i / (p.rd1 * p.rd0)) * p.rs[0] +
                       (int64_t)(i / p.rd1 % p.rd0) * p.rs[1] + (int64_t)(i % p.rd1) * p.rs[2];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int cc = min(c, n - 1);
      const double v = p.A[ro + (int64_t)(cc / p.cd) * p.cs[0] + (int64_t)(cc % p.cd) * p.cs[1]];
      w[r][c] = (c < n && tid + NT * r < m) ? v : 0.0;
    }
  }
  // sums of g over the workgroup: lane l gets that of value l mod 16; one
  // barrier, buffers in turn
  auto sum_all = [&](const double (&g)[NC], int buf) {
    double k[NC / 4];
    sum64_many<NC>(g, k);
    const int at = lanes_of(lane);
#pragma unroll
    for (int t = 0; t < NC / 4; ++t)
      if ((lane & 15) == t) part[buf][wave][4 * t + at] = k[t];
    __syncthreads();
    double s = 0.0;
    const int c = min(lane & 15, NC - 1);
#pragma unroll
    for (int x = 0; x < NWV; ++x) s += part[buf][x][c];
    return s;
  };
  double tau[NC];
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    tau[j] = 0.0;
    if (j >= kmax) continue;
    double g[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) g[c] = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const double x = tid + NT * r > j ? w[r][j] : 0.0;
#pragma unroll
      for (int c = j; c < NC; ++c) g[c] = fma(x, w[r][c], g[c]);
    }
    if (tid == j) {
#pragma unroll
      for (int c = j; c < NC; ++c) rowj[j & 1][c] = w[0][c];
    }
    const double gs = sum_all(g, j & 1);
    const double row = rowj[j & 1][min(lane & 15, NC - 1)];
    const double alpha = lane_value(row, j), xnorm2 = lane_value(gs, j);
    double beta = alpha, t = 0.0, scal = 0.0;
    if (xnorm2 > 0.0) {
      beta = -copysign(sqrt(alpha * alpha + xnorm2), alpha);
      t = (beta - alpha) / beta;
      scal = 1.0 / (alpha - beta);
    }
    tau[j] = t;
    const double wl = t * fma(scal, gs, row);
    double v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = tid + NT * r;
      v[r] = i > j ? w[r][j] * scal : (i == j ? 1.0 : 0.0);
      w[r][j] = i > j ? v[r] : (i == j ? beta : w[r][j]);
    }
#pragma unroll
    for (int c = j + 1; c < NC; ++c) {
      const double x = lane_value(wl, c);
#pragma unroll
      for (int r = 0; r < R; ++r) w[r][c] = fma(-v[r], x, w[r][c]);
    }
  }
  // R (n x n, upper; rows beyond kmax are zero): row i is in thread i
  if (tid < n) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if (c < n) p.R[tid * n + c] = (tid <= c && tid < kmax) ? w[0][c] : 0.0;
  }
  if (p.Q == nullptr) return;
  // thin Q = H_0 ... H_{kmax-1} I[:, :kmax]  (m x kmax, leading dimension n)
  double q[R][NC];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < NC; ++c) q[r][c] = tid + NT * r == c ? 1.0 : 0.0;
  int buf = kmax & 1;  // the factorisation's last buffer was the other one
#pragma unroll
  for (int j = NC - 1; j >= 0; --j) {
    if (j >= kmax) continue;
    const double t = tau[j];
    if (t == 0.0) continue;
    double g[NC], v[R];
#pragma unroll
    for (int c = 0; c < NC; ++c) g[c] = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = tid + NT * r;
      v[r] = i > j ? w[r][j] : (i == j ? 1.0 : 0.0);
#pragma unroll
      for (int c = j; c < NC; ++c) g[c] = fma(v[r], q[r][c], g[c]);
    }
    const double wl = t * sum_all(g, buf);
    buf ^= 1;
#pragma unroll
    for (int c = j; c < NC; ++c) {
      const double x = lane_value(wl, c);
#pragma unroll
      for (int r = 0; r < R; ++r) q[r][c] = fma(-v[r], x, q[r][c]);
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if (c < n && tid + NT * r < m) p.Q[(int64_t)(tid + NT * r) * n + c] = c < kmax ? q[r][c] : 0.0;
}

// ---------------------------------------------------------------------------
// SVD of a tiny dense n x n matrix (n <= 32), A V = U S with S descending:
// Householder QR of the columns in falling order of their norms, A P = Q R,
// then one-sided (Hestenes) Jacobi on the columns of R^T, which the graded
// rows of R leave in 6 - 8 sweeps where the columns of A itself take 8 to 19:
// R^T W = Y S, so U = Q W and V = P Y.  Half a wave per column pair (lane i
// holds row i), round-robin pair ordering; a pair is rotated while
// |a_p . a_q| > 1e-15 * ||a_p|| ||a_q||.  Bound by instruction issue: one
// barrier a round, the three inner products summed by lane exchanges without
// LDS, the rotation by refined hardware reciprocals (24 x 24, graded: 111
// us; 153 us with a wave a pair, 270 us without the factorisation as well,
// 430 us with shuffles and full divisions).
// ---------------------------------------------------------------------------
constexpr int SVD_NT = 512;  // at most: half a wave for each of n / 2 pairs

// the tangent of the rotation where squares would leave the range of a double
__device__ __noinline__ double tiny_tangent(double dl, double ga) {
  const double zeta = dl / (2.0 * ga);
  return (zeta >= 0.0 ? 1.0 : -1.0) / (fabs(zeta) + sqrt(1.0 + zeta * zeta));
}

// order[]: 0..n-1 by falling nrm (the identity where NaNs leave ranks empty)
__device__ __forceinline__ void falling_order(const double* nrm, int* order, int n) {
  const int tid = threadIdx.x;
  if (tid < n) order[tid] = tid;
  __syncthreads();
  if (tid < n) {
    int rank = 0;
    for (int j = 0; j < n; ++j) rank += (nrm[j] > nrm[tid]) || (nrm[j] == nrm[tid] && j < tid);
    order[rank] = tid;
  }
  __syncthreads();
}

__global__ __launch_bounds__(SVD_NT) void svd_small_kernel(const double* __restrict__ A, int n,
                                                           double* __restrict__ U,
                                                           double* __restrict__ s,
                                                           double* __restrict__ V,
                                                           int64_t batch_stride) {
  // workgroup b decomposes problem b: matrices batch_stride doubles apart,
  // singular values n apart
  A += blockIdx.x * batch_stride;
  U += blockIdx.x * batch_stride;
  V += blockIdx.x * batch_stride;
  s += (int64_t)blockIdx.x * n;
  constexpr int LD = kSvdMaxN + 1;
  __shared__ double a[kSvdMaxN][LD];   // columns of A P, then of R^T
  __shared__ double vh[kSvdMaxN][LD];  // columns of A, then the reflectors, zero above their one
  __shared__ double v[kSvdMaxN][LD];   // columns of W
  __shared__ double nrm[kSvdMaxN], tau[kSvdMaxN];
  __shared__ int order[kSvdMaxN], perm[kSvdMaxN];
  const int tid = threadIdx.x, lane = tid & 63, l = lane & 31, nt = blockDim.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // a unit (half a wave) has one pair and up to two columns, unit + {0, units}
  const int unit = tid >> 5, units = nt >> 5;
  const int nn = n + (n & 1);
  auto norms = [&](const double (*x)[LD]) {
    for (int c0 = 0; c0 < n; c0 += units) {
      const int c = c0 + unit;
      const double y = x[min(c, n - 1)][l], ss = sum32(y * y);
      if (l == 0 && c < n) nrm[c] = sqrt(ss);
    }
    __syncthreads();
  };
  for (int e = tid; e < kSvdMaxN * 32; e += nt) {
    const int c = e & 31, r = e >> 5;
    vh[c][r] = (c < n && r < n) ? A[r * n + c] : 0.0;
    v[c][r] = (r == c) ? 1.0 : 0.0;
  }
  __syncthreads();
  norms(vh);
  falling_order(nrm, perm, n);
  for (int c = unit; c < n; c += units) a[c][l] = vh[perm[c]][l];
  // QR: the wave of column j + 1 prepares its reflector behind the update by
  // reflector j
  auto reflector = [&](int j) {
    const double x = a[j][l];
    const double xnorm2 = sum32(l > j ? x * x : 0.0), alpha = lane_value(x, j);
    double beta = alpha, t = 0.0, scal = 0.0;
    if (xnorm2 > 0.0) {
      beta = -copysign(sqrt(alpha * alpha + xnorm2), alpha);
      t = (beta - alpha) / beta;
      scal = 1.0 / (alpha - beta);
    }
    vh[j][l] = l > j ? x * scal : (l == j ? 1.0 : 0.0);
    a[j][l] = l > j ? 0.0 : (l == j ? beta : x);
    if (lane == 0) tau[j] = t;
  };
  __syncthreads();  // vh read by all
  if (wave == 0) reflector(0);
  __syncthreads();
  for (int j = 0; j + 1 < n; ++j) {
    const double h = vh[j][l], t = tau[j];
    for (int c0 = j + 1 >= units ? units : 0; c0 < n; c0 += units) {
      const int c = c0 + unit;
      const double x = a[min(c, n - 1)][l], y = fma(-t * sum32(h * x), h, x);
      if (c > j && c < n) a[c][l] = y;
    }
    const int own = j + 1 >= units ? j + 1 - units : j + 1;
    if (wave == own >> 1) reflector(j + 1);
    __syncthreads();
  }
  // a <- R^T: column c is row c of R
  const int c1 = min(unit + units, n - 1);
  const double t0 = a[l][min(unit, n - 1)], t1 = a[l][c1];
  __syncthreads();
  if (unit < n) a[unit][l] = l < n && l >= unit ? t0 : 0.0;
  if (unit + units < n) a[c1][l] = l < n && l >= c1 ? t1 : 0.0;
  __syncthreads();
  for (int sweep = 0; sweep < 60; ++sweep) {
    int rot = 0;
    for (int r = 0; r < nn - 1; ++r) {
      int x = nn - 1, y = r;
      if (unit > 0) {
        x = r + unit;
        if (x >= nn - 1) x -= nn - 1;
        y = r - unit;
        if (y < 0) y += nn - 1;
      }
      const int p = min(x, y), q = max(x, y);
      const bool pair = unit < nn / 2 && q < n;
      const int pc = pair ? p : 0, qc = pair ? q : 0;
      const double ap = a[pc][l], aq = a[qc][l], vp = v[pc][l], vq = v[qc][l];
      // row 0 of the half sums one value, row 1 the other
      const double n2 = sum16(swap16_sum(ap * ap, aq * aq));
      const double ga = sum32(ap * aq);
      double al, be;
      swap16(n2, n2, al, be);
      const double ab = al * be;
      // in squares unless they leave the range of a double
      if (pair && ga != 0.0 &&
          (ab > 1e-200 ? ga * ga > 1e-30 * ab : fabs(ga) > 1e-15 * sqrt(ab))) {
        // t = sgn(zeta) / (|zeta| + sqrt(1 + zeta^2)), zeta = (be - al) / (2 ga)
        const double dl = be - al, h2 = fma(dl, dl, 4.0 * ga * ga);
        const double t = h2 > 1e-280 && h2 < 1e280
                             ? copysign(2.0, dl) * ga * rcp_nr(fabs(dl) + h2 * rsqrt_nr(h2))
                             : tiny_tangent(dl, ga);
        const double c = rsqrt_nr(fma(t, t, 1.0)), sn = c * t;
        a[p][l] = c * ap - sn * aq;
        a[q][l] = sn * ap + c * aq;
        v[p][l] = c * vp - sn * vq;
        v[q][l] = sn * vp + c * vq;
        // cosines and angles below 1e-9 all through a sweep leave products of two
        // of them, below 1e-17: the sweep that would find nothing is not run
        rot |= ga * ga > 1e-18 * ab || fabs(t) > 1e-9;
      }
      __syncthreads();
    }
    if (!__syncthreads_or(rot)) break;
  }
  norms(a);
  falling_order(nrm, order, n);
  // U = Q W, a column a unit; V = P Y
  for (int k0 = 0; k0 < n; k0 += units) {
    const int k = k0 + unit, c = order[min(k, n - 1)];
    double u = v[c][l];
    for (int j = n - 1; j >= 0; --j) {
      const double h = vh[j][l];
      u = fma(-tau[j] * sum32(h * u), h, u);
    }
    if (k < n && l < n) {
      U[l * n + k] = u;
      V[perm[l] * n + k] = nrm[c] > 0.0 ? a[c][l] / nrm[c] : 0.0;
    }
    if (k < n && l == 0) s[k] = nrm[c];
  }
}

// ---------------------------------------------------------------------------
// small elementwise helpers
// ---------------------------------------------------------------------------
// M[i][j] = M[j][i] for i < j: the symmetric matrix that an eigensolver
// reading only the lower triangle sees (LAPACK's and torch's UPLO='L').
__global__ void lower_to_full_kernel(double* M, int n) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < (int64_t)n * n;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int i = (int)(e / n), j = (int)(e % n);
    if (i < j) M[e] = M[(int64_t)j * n + i];
  }
}

__global__ void add_diag_kernel(double* M, int n, double shift) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    M[(int64_t)i * n + i] += shift;
}

// X[r][z] = Z[r][z] * sqrt(w[z])
__global__ void scale_sqrt_kernel(const double* __restrict__ Z, const double* __restrict__ w,
                                  int rows, int cols, double* __restrict__ X) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < (int64_t)rows * cols;
       e += (int64_t)gridDim.x * blockDim.x)
    X[e] = Z[e] * sqrt(w[e % cols]);
}

// pinv = V diag(1/s, s > atol) U^T  (U m x n, V n x n; result n x m)
__global__ void pinv_finish_kernel(const double* __restrict__ U, const double* __restrict__ s,
                                   const double* __restrict__ V, int m, int n, double atol,
                                   double* __restrict__ P) {
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < n * m; e += gridDim.x * blockDim.x) {
    const int i = e / m, j = e % m;
    double acc = 0.0;
    for (int k = 0; k < n; ++k)
      if (s[k] > atol) acc += V[i * n + k] * (1.0 / s[k]) * U[j * n + k];
    P[e] = acc;
  }
}

// finalize_reduced_tensors scaling: s' = sqrt(s[:bD] / ||s||);
// r1n[a][u] = U[a][u] s'_u (U n x n), r2n[v][b] = s'_v Vt[v][b] = s'_v V[b][v]
__global__ void finalize_scale_kernel(const double* __restrict__ U, const double* __restrict__ s,
                                      const double* __restrict__ V, int n, int bD,
                                      double* __restrict__ r1n, double* __restrict__ r2n) {
  __shared__ double nrm;
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int k = 0; k < n; ++k) t += s[k] * s[k];
    nrm = sqrt(t);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < n * bD; e += blockDim.x) {
    const int a = e / bD, u = e % bD;
    const double sp = sqrt(s[u] / nrm);
    r1n[a * bD + u] = U[a * n + u] * sp;
    r2n[u * n + a] = sp * V[a * n + u];
  }
}

// Bond-index sign gauge shared with the oracle: sign(sum_i w_i f[u][i]) > 0
// with f[u][(y, p)] = a1r[y][u][p] and w_i = 1 + frac(i * 0.6180339887498949).
__global__ void bond_gauge_kernel(double* __restrict__ a1r, double* __restrict__ a2r, int nD1,
                                  int nD2, int bD, int pD) {
  __shared__ double red[4];
  __shared__ double sgn;
  const int u = blockIdx.x;
  double acc = 0.0;
  for (int i = threadIdx.x; i < nD1 * pD; i += blockDim.x) {
    const int y = i / pD, p = i % pD;
    const double x = (double)i * 0.6180339887498949;
    acc += (1.0 + (x - floor(x))) * a1r[(y * bD + u) * pD + p];
  }
  const double t = block_sum(acc, red);
  if (threadIdx.x == 0) sgn = (t < 0.0) ? -1.0 : 1.0;
  __syncthreads();
  for (int i = threadIdx.x; i < nD1 * pD; i += blockDim.x) {
    const int y = i / pD, p = i % pD;
    a1r[(y * bD + u) * pD + p] *= sgn;
  }
  for (int i = threadIdx.x; i < nD2 * pD; i += blockDim.x) {
    const int x = i / pD, q = i % pD;
    a2r[(x * bD + u) * pD + q] *= sgn;
  }
}

// Simple update: out = A * prod_legs w_leg (or 1 / max(w_leg, cutoff) when
// invert) over the four bond legs; a null weight vector is all ones.
__global__ void lambda_scale_kernel(const double* __restrict__ A, double* __restrict__ out,
                                    LambdaLegs w, int D, int d, int invert, double cutoff) {
  const int64_t n = (int64_t)D * D * D * D * d;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n;
       e += (int64_t)gridDim.x * blockDim.x) {
    int64_t r = e / d;
    double f = 1.0;
    for (int leg = 3; leg >= 0; --leg) {
      const int i = (int)(r % D);
      r /= D;
      if (w.v[leg] != nullptr) {
        const double x = w.v[leg][i];
        f *= invert ? 1.0 / fmax(x, cutoff) : x;
      }
    }
    out[e] = A[e] * f;
  }
}

// Simple-update split of the gated bond matrix (simple_update.py:53-61):
// lt = sqrt(S[:bD] / ||S[:bD]||), a1r[y][a][p] = U[(y,p)][a] lt[a],
// a2r[x][a][q] = V[(x,q)][a] lt[a]  (U, V n x n with n = nD pD).
__global__ void su_split_kernel(const double* __restrict__ U, const double* __restrict__ S,
                                const double* __restrict__ V, int nD, int bD, int pD,
                                double* __restrict__ a1r, double* __restrict__ a2r,
                                double* __restrict__ lt) {
  __shared__ double nrm;
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int a = 0; a < bD; ++a) t += S[a] * S[a];
    nrm = sqrt(t);
  }
  __syncthreads();
  const int n = nD * pD;
  for (int e = threadIdx.x; e < nD * bD * pD; e += blockDim.x) {
    const int y = e / (bD * pD), a = (e / pD) % bD, p = e % pD;
    const double l = sqrt(S[a] / nrm);
    a1r[e] = U[(y * pD + p) * n + a] * l;
    a2r[e] = V[(y * pD + p) * n + a] * l;
  }
  for (int a = threadIdx.x; a < bD; a += blockDim.x) lt[a] = sqrt(S[a] / nrm);
}

// ---------------------------------------------------------------------------
// Persistent ALS solver (ALSSolver.solve / solve_torch, als_solver.py:34-82,
// with build_s1/s2/r1/r2, solve_ar and calculate_cost, :148-260), one
// workgroup, the whole sweep loop and its stopping rule on the device.
//
// Index names follow the reference: n12[y][x][Y][X], a12g[y][x][p][q],
// a1r[y][u][p], a2r[x][v][q].  Per sweep:
//   R1[(Y,U),(y,u)] = sum_{x,X,Q} n12[y,x,Y,X] a2r[x,u,Q] a2r[X,U,Q]
//   S1[(Y,U),p]     = sum_{X,Q}   n12g[Y,X,p,Q] a2r[X,U,Q]
//   a1r = solve(sym(R1) + eps max|R1| I, S1)   (Cholesky; LU fallback)
// and the mirror image for a2r; then the cost
//   d2 - 2 d3,  d2 = <a12n|N|a12n>, d3 = <a12n|N|a12g>, a12n = a1r a2r.
// Stops after sweep i (0-based) when |d2 - d1| / |d1| < tol and i > 1.
// ---------------------------------------------------------------------------
constexpr int ALS_NT = 256;

struct AlsShared {
  double* R;     // nR x nR
  double* S;     // nR x d
  double* a1;    // nD x D x d
  double* a2;
  double* T;     // nD x nD x D x d for each of grp outer indices of the R build
  double* n12g;  // nD^2 d^2
  double* a12n;  // nD^2 d^2
  double* red;   // ALS_NT/64
};

typedef double als_d4 __attribute__((ext_vector_type(4)));

// na = N x for x[(y,x)][pq] in LDS (nD^2 x d^2): 16 x 16 tiles on the matrix
// cores, a row tile a wave at a time; take(e, value) gets element e of na.
template <class F>
__device__ __forceinline__ void als_apply_norm(const double* __restrict__ n12,
                                               const double* __restrict__ x, int nD, int d2,
                                               F&& take) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, m = lane & 15, kq = lane >> 4;
  const int n2 = nD * nD, mt = (n2 + 15) / 16, nt = (d2 + 15) / 16;
  for (int t = wave; t < mt * nt; t += ALS_NT / 64) {
    const int row = t % mt * 16, cl = t / mt * 16 + m, cc = min(cl, d2 - 1);
    const double* pa = n12 + min(row + m, n2 - 1);
    als_d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 8
    for (int k0 = 0; k0 < n2; k0 += 4) {
      const int k = min(k0 + kq, n2 - 1);
      const double av = pa[(int64_t)k * n2], bv = x[k * d2 + cc];
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(k0 + kq < n2 ? av : 0.0, bv, acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = row + kq + 4 * r;
      if (i < n2 && cl < d2) take(i * d2 + cl, acc[r]);
    }
  }
}

// Build R and S for the tensor of side ``side`` from ``other`` (the fixed one),
// ``grp`` outer indices a at a time (as many as T holds).  Both contractions run
// on the matrix cores, operands straight from memory and LDS: on 256 threads'
// vector units every product cost a load of its own (nD = 12, the whole call of a
// D=6 bond: 1530 -> 675 us).
__device__ void als_build(const AlsShared& sh, const double* __restrict__ n12, int side, int nD,
                          int D, int d, int grp, const double* other) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, m = lane & 15, kq = lane >> 4;
  const int nR = nD * D, Dd = D * d, n2 = nD * nD;
  const int mt = (n2 + 15) / 16, nt = (Dd + 15) / 16;
  for (int a0 = 0; a0 < nD; a0 += grp) {
    const int ga = min(grp, nD - a0);
    // T[a][A][B][uQ] = sum_b N(a,b,A,B) other[b][uQ]; N is contiguous in (A, B)
    // on side 0, in (B, A) on side 1
    for (int t0 = wave * 2; t0 < ga * mt * nt; t0 += ALS_NT / 32) {
      als_d4 acc[2];
      const double *pa[2], *pb[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int t = min(t0 + h, ga * mt * nt - 1), g = t / (mt * nt), row = t % mt * 16;
        acc[h] = als_d4{0.0, 0.0, 0.0, 0.0};
        pa[h] = n12 + (int64_t)(side == 0 ? (a0 + g) * nD : a0 + g) * n2 + min(row + m, n2 - 1);
        pb[h] = other + min(t / mt % nt * 16 + m, Dd - 1);
      }
      const int64_t sb = side == 0 ? n2 : (int64_t)nD * n2;  // from b to b + 1
#pragma unroll 3
      for (int k0 = 0; k0 < nD; k0 += 4) {
        const int k = min(k0 + kq, nD - 1);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const double av = pa[h][k * sb], bv = pb[h][k * Dd];
          acc[h] = __builtin_amdgcn_mfma_f64_16x16x4f64(k0 + kq < nD ? av : 0.0, bv, acc[h], 0, 0, 0);
        }
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int t = t0 + h, g = t / (mt * nt), row = t % mt * 16, cl = t / mt % nt * 16 + m;
        if (t >= ga * mt * nt || cl >= Dd) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = row + kq + 4 * r;
          const int ab = side == 0 ? i : i % nD * nD + i / nD;
          if (i < n2) sh.T[((int64_t)g * n2 + ab) * Dd + cl] = acc[h][r];
        }
      }
    }
    __syncthreads();
    // R[(A,U),(a,u)] = sum_{B,Q} T[a][A][B][u][Q] other[B][U][Q], rows (A, u), columns U
    const int rt = (nR + 15) / 16, ut = (D + 15) / 16, K = nD * d;
    for (int t = wave; t < ga * rt * ut; t += ALS_NT / 64) {
      const int g = t / (rt * ut), row = t % rt * 16, cl = t / rt % ut * 16 + m;
      const int i = min(row + m, nR - 1), U = min(cl, D - 1);
      const double* pt = sh.T + (int64_t)g * n2 * Dd + i / D * nD * Dd + i % D * d;
      als_d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 2
      for (int k0 = 0; k0 < K; k0 += 4) {
        const int k = min(k0 + kq, K - 1), B = k / d, Q = k - B * d;
        const double av = pt[B * Dd + Q], bv = other[(B * D + U) * d + Q];
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(k0 + kq < K ? av : 0.0, bv, acc, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int x = row + kq + 4 * r, A = x / D, u = x % D;
        if (x < nR && cl < D) sh.R[(int64_t)(A * D + cl) * nR + (a0 + g) * D + u] = acc[r];
      }
    }
    __syncthreads();
  }
  // S[(A,U)][p] = sum_{B,Q} G(A,B,p,Q) other[B][U][Q]
  const int d2 = d * d;
  for (int e = tid; e < nR * d; e += ALS_NT) {
    const int A = e / (D * d), U = (e / d) % D, p = e % d;
    double acc = 0.0;
    for (int B = 0; B < nD; ++B)
      for (int Q = 0; Q < d; ++Q) {
        const double g = side == 0 ? sh.n12g[(A * nD + B) * d2 + p * d + Q]
                                   : sh.n12g[(B * nD + A) * d2 + Q * d + p];
        acc += g * other[(B * D + U) * d + Q];
      }
    sh.S[e] = acc;
  }
  __syncthreads();
}

__device__ double block_max(double v, double* red) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t = fmax(t, red[w]);
  return t;
}

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ALS system through the pseudo-inverse (als_solver.py:228-230:
// pinv(R, hermitian=True, rcond=eps) @ S): R <- (R + R^T)/2 (no shift),
// R = V diag(lam) V^T by cyclic two-sided Jacobi with round-robin parallel
// pairs (R in LDS, V in the global scratch), then S <- V diag(w) V^T S with
// w_i = 1/lam_i for |lam_i| > eps * max|lam|, else 0.
__device__ void als_pinv_solve(const AlsShared& sh, int nR, int d, double eps,
                               double* __restrict__ V) {
  const int tid = threadIdx.x;
  double* R = sh.R;
  double* S = sh.S;
  __shared__ double rc[128], rs[128];
  __shared__ int rp[128], rq[128];
  __shared__ int s_rot;
  for (int e = tid; e < nR * nR; e += ALS_NT) {
    const int i = e / nR, j = e % nR;
    if (i < j) {
      const double v = 0.5 * (R[i * nR + j] + R[j * nR + i]);
      R[i * nR + j] = v;
      R[j * nR + i] = v;
    }
    V[e] = (i == j) ? 1.0 : 0.0;
  }
  __syncthreads();
  const int n = nR + (nR & 1);  // padding index n - 1 (odd nR) never rotates
  const int half = n / 2;
  for (int sweep = 0; sweep < 60; ++sweep) {
    if (tid == 0) s_rot = 0;
    __syncthreads();
    for (int round = 0; round < n - 1; ++round) {
      // circle method: index n - 1 fixed, the others rotate
      for (int a = tid; a < half; a += ALS_NT) {
        int p = (a == 0) ? n - 1 : (round + a) % (n - 1);
        int q = (round - a + (n - 1)) % (n - 1);
        if (a == 0) q = round;
        if (p > q) { const int t = p; p = q; q = t; }
        double c = 1.0, sn = 0.0;
        if (q < nR) {
          const double app = R[p * nR + p], aqq = R[q * nR + q], apq = R[p * nR + q];
          if (fabs(apq) > 1e-15 * sqrt(fabs(app * aqq)) && apq != 0.0) {
            const double zeta = (aqq - app) / (2.0 * apq);
            const double t = (zeta >= 0.0 ? 1.0 : -1.0) / (fabs(zeta) + sqrt(1.0 + zeta * zeta));
            c = 1.0 / sqrt(1.0 + t * t);
            sn = c * t;
            s_rot = 1;
          }
        }
        rc[a] = c; rs[a] = sn; rp[a] = p; rq[a] = q;
      }
      __syncthreads();
      // rows: R[p,:], R[q,:] <- c R[p,:] - s R[q,:], s R[p,:] + c R[q,:]
      for (int e = tid; e < half * nR; e += ALS_NT) {
        const int a = e / nR, k = e % nR;
        const int p = rp[a], q = rq[a];
        if (q >= nR || rs[a] == 0.0) continue;
        const double c = rc[a], sn = rs[a];
        const double x = R[p * nR + k], y = R[q * nR + k];
        R[p * nR + k] = c * x - sn * y;
        R[q * nR + k] = sn * x + c * y;
      }
      __syncthreads();
      // columns of R and V
      for (int e = tid; e < half * nR; e += ALS_NT) {
        const int a = e / nR, k = e % nR;
        const int p = rp[a], q = rq[a];
        if (q >= nR || rs[a] == 0.0) continue;
        const double c = rc[a], sn = rs[a];
        const double x = R[k * nR + p], y = R[k * nR + q];
        R[k * nR + p] = c * x - sn * y;
        R[k * nR + q] = sn * x + c * y;
        const double vx = V[k * nR + p], vy = V[k * nR + q];
        V[k * nR + p] = c * vx - sn * vy;
        V[k * nR + q] = sn * vx + c * vy;
      }
      __syncthreads();
    }
    if (!s_rot) break;
    __syncthreads();
  }
  // S <- V diag(w) V^T S; T = V^T S staged in R's off-diagonal-free copy
  double mx = 0.0;
  for (int i = tid; i < nR; i += ALS_NT) mx = fmax(mx, fabs(R[i * nR + i]));
  mx = block_max(mx, sh.red);
  double* T = R;  // the eigenvalues are read once below, before T overwrites row 0
  __shared__ double lam[256];
  for (int i = tid; i < nR; i += ALS_NT) lam[i] = R[i * nR + i];
  __syncthreads();
  for (int e = tid; e < nR * d; e += ALS_NT) {
    const int i = e / d, c = e % d;
    double acc = 0.0;
    for (int k = 0; k < nR; ++k) acc += V[k * nR + i] * S[k * d + c];
    const double li = lam[i];
    T[e] = (fabs(li) > eps * mx) ? acc / li : 0.0;
  }
  __syncthreads();
  for (int e = tid; e < nR * d; e += ALS_NT) {
    const int i = e / d, c = e % d;
    double acc = 0.0;
    for (int k = 0; k < nR; ++k) acc += V[i * nR + k] * T[k * d + c];
    S[e] = acc;
  }
  __syncthreads();
}

// The elimination behind als_solve_system with the lower triangle in registers:
// thread (ti, tj) of 16 x 16 holds rows ti + 16 r and columns tj + 16 c, r >= c
// < RC.  A step publishes its column and its row of S (one barrier, two buffers
// in turn) and every thread subtracts the products of the column with itself
// over the pivot from its part, right-hand sides included; columns stay
// unscaled (L D).  On return R's lower triangle holds L D, dinv 1 / D and S the
// forward-substituted right-hand sides.  False if a pivot was not positive: S
// and R's upper triangle are then untouched.
template <int RC>
__device__ bool als_eliminate(double* R, double* S, int nR, int d, double shift,
                              double* __restrict__ pub, double* dinv) {
  constexpr int PB = 16 * RC + 8;  // a published column and the row of S
  const int tid = threadIdx.x, ti = tid >> 4, tj = tid & 15;
  double a[RC][RC], s[RC];
#pragma unroll
  for (int r = 0; r < RC; ++r) {
    const int i = ti + 16 * r;
#pragma unroll
    for (int c = 0; c <= r; ++c) {
      const int k = tj + 16 * c;
      const double v = (i < nR && k < nR && k <= i) ? R[k * nR + i] : 0.0;
      a[r][c] = i == k ? v + shift : v;
    }
    s[r] = (i < nR && tj < d) ? S[i * d + tj] : 0.0;
  }
#pragma unroll
  for (int cj = 0; cj < RC; ++cj) {
#pragma unroll 1
    for (int jj = 0; jj < 16; ++jj) {
      const int j = 16 * cj + jj;
      if (j >= nR) break;
      double* col = pub + (j & 1) * PB;
      if (tj == jj) {
#pragma unroll
        for (int r = cj; r < RC; ++r) {
          const int i = ti + 16 * r;
          col[i] = a[r][cj];
          if (i >= j && i < nR) R[i * nR + j] = a[r][cj];
        }
      }
      if (ti == jj && tj < d) col[16 * RC + tj] = s[cj];
      __syncthreads();
      const double piv = col[j];
      if (!(piv > 0.0)) return false;
      const double inv = 1.0 / piv;
      if (tid == 0) dinv[j] = inv;
      double ck[RC];
#pragma unroll
      for (int c = cj; c < RC; ++c) ck[c] = tj + 16 * c > j ? col[tj + 16 * c] * inv : 0.0;
      const double sk = tj < d ? col[16 * RC + tj] * inv : 0.0;
#pragma unroll
      for (int r = cj; r < RC; ++r) {
        const double x = ti + 16 * r > j ? col[ti + 16 * r] : 0.0;
#pragma unroll
        for (int c = cj; c <= r; ++c) a[r][c] = fma(-x, ck[c], a[r][c]);
        s[r] = fma(-x, sk, s[r]);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < RC; ++r) {
    const int i = ti + 16 * r;
    if (i < nR && tj < d) S[i * d + tj] = s[r];
  }
  __syncthreads();
  return true;
}

// Solve (sym(R) + eps max|R| I) X = S in place (X -> S).  Returns (block-
// uniform) 0, 1 if a pivot was not positive and partial-pivoting elimination was
// used, 2 if that found R singular.  The factorisation was one wave's walk
// through LDS and most of a sweep; on all 256 threads it is bound by the step's
// round trip (nR = 72, the whole call of a D=6 bond: 2440 -> 1530 us).
constexpr int kAlsMaxTiles = 9;  // nR <= 144 (LDS holds less)
template <int RC>
__device__ int als_solve_system(const AlsShared& sh, int nR, int d, double eps, int* flag) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  __shared__ double pub[2 * (16 * RC + 8)], dinv[16 * RC];
  double* R = sh.R;
  double* S = sh.S;
  // the symmetric part goes to the upper triangle
  double mx = 0.0;
  for (int e = tid; e < nR * nR; e += ALS_NT) {
    const int i = e / nR, j = e % nR;
    if (i <= j) {
      const double v = 0.5 * (R[i * nR + j] + R[j * nR + i]);
      R[i * nR + j] = v;
      mx = fmax(mx, fabs(v));
    }
  }
  mx = block_max(mx, sh.red);
  const double shift = eps * mx;
  // the lower triangle takes the factor, the diagonal with it
  double diag = tid < nR ? R[tid * nR + tid] + shift : 0.0;
  if (tid == 0) *flag = 0;
  __syncthreads();
  if (als_eliminate<RC>(R, S, nR, d, shift, pub, dinv)) {
    // D L^T x = S, a right-hand side a wave: lane l holds rows l, l + 64, l + 128
    for (int c = wave; c < d; c += ALS_NT / 64) {
      double x[3], w[3];
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        const int i = lane + 64 * t;
        x[t] = i < nR ? S[i * d + c] : 0.0;
        w[t] = i < nR ? dinv[i] : 0.0;
      }
#pragma unroll
      for (int t = 2; t >= 0; --t) {
#pragma unroll 4
        for (int k = min(nR, 64 * t + 64) - 1; k >= 64 * t; --k) {
          const double xk = lane_value(x[t] * w[t], k - 64 * t);
#pragma unroll
          for (int h = 0; h <= t; ++h) {
            const int i = lane + 64 * h;
            const double l = R[k * nR + min(i, k)];
            x[h] = fma(-(i < k ? l : 0.0), xk, x[h]);
          }
        }
      }
#pragma unroll
      for (int t = 0; t < 3; ++t)
        if (lane + 64 * t < nR) S[(lane + 64 * t) * d + c] = x[t] * w[t];
    }
    __syncthreads();
    return 0;
  }
  // LU with partial pivoting on the regularised system
  __syncthreads();
  for (int e = tid; e < nR * nR; e += ALS_NT) {
    const int i = e / nR, j = e % nR;
    if (i < j) R[j * nR + i] = R[i * nR + j];
  }
  if (tid < nR) R[tid * nR + tid] = diag;
  if (tid == 0) *flag = 1;
  __syncthreads();
  if (tid < 64) {
    int singular = 0;
    for (int j = 0; j < nR; ++j) {
      // pivot search over rows j..nR-1
      double best = -1.0;
      int bi = j;
      for (int i = j + lane; i < nR; i += 64) {
        const double v = fabs(R[i * nR + j]);
        if (v > best) { best = v; bi = i; }
      }
      for (int o = 32; o > 0; o >>= 1) {
        const double ob = __shfl_xor(best, o);
        const int oi = __shfl_xor(bi, o);
        if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
      }
      if (!(best > 0.0)) { singular = 1; break; }
      wave_sync();
      if (bi != j) {
        for (int c = lane; c < nR; c += 64) {
          const double t = R[j * nR + c];
          R[j * nR + c] = R[bi * nR + c];
          R[bi * nR + c] = t;
        }
        if (lane < d) {
          const double t = S[j * d + lane];
          S[j * d + lane] = S[bi * d + lane];
          S[bi * d + lane] = t;
        }
      }
      wave_sync();
      const double pjj = R[j * nR + j];
      for (int i = j + 1 + lane; i < nR; i += 64) {
        const double f = R[i * nR + j] / pjj;
        for (int c = j + 1; c < nR; ++c) R[i * nR + c] -= f * R[j * nR + c];
        for (int c = 0; c < d; ++c) S[i * d + c] -= f * S[j * d + c];
      }
      wave_sync();
    }
    if (!singular) {
      for (int k = nR - 1; k >= 0; --k) {
        const double ukk = R[k * nR + k];
        wave_sync();
        if (lane < d) S[k * d + lane] /= ukk;
        wave_sync();
        for (int i = lane; i < k; i += 64) {
          const double uik = R[i * nR + k];
          for (int c = 0; c < d; ++c) S[i * d + c] -= uik * S[k * d + c];
        }
        wave_sync();
      }
    } else if (lane == 0) {
      *flag = 2;
    }
  }
  __syncthreads();
  return *flag;
}

// cost = d2 - 2 d3 of the current (a1, a2)
__device__ double als_cost(const AlsShared& sh, const double* __restrict__ n12, int nD, int D,
                           int d) {
  const int tid = threadIdx.x;
  const int d2 = d * d, nE = nD * nD * d2;
  for (int e = tid; e < nE; e += ALS_NT) {
    const int y = e / (nD * d2), x = (e / d2) % nD, p = (e / d) % d, q = e % d;
    double acc = 0.0;
    for (int u = 0; u < D; ++u) acc += sh.a1[(y * D + u) * d + p] * sh.a2[(x * D + u) * d + q];
    sh.a12n[e] = acc;
  }
  __syncthreads();
  double part = 0.0;
  als_apply_norm(n12, sh.a12n, nD, d2, [&](int e, double na) {
    part += na * sh.a12n[e] - 2.0 * sh.n12g[e] * sh.a12n[e];
  });
  return block_sum(part, sh.red);
}

// RC: the elimination's tiles (nR <= 16 RC), 0 for the pseudo-inverse: one kernel
// each, for what the largest holds in registers would halve a batch of small
// problems' workgroups a CU (4000 of D=3: 1.26 ms, 3.2 ms with one kernel for all,
// 2.1 ms with one wave factorising; 1000 of D=6: 2.5, 4.1, 8.0)
template <int RC>
__global__ __launch_bounds__(ALS_NT) void als_kernel(const double* __restrict__ n12,
                                                     const double* __restrict__ a12g,
                                                     double* __restrict__ a1r,
                                                     double* __restrict__ a2r, int nD, int D,
                                                     int d, int niter, double tol, double eps,
                                                     double* __restrict__ gwork,
                                                     double* __restrict__ out_cost,
                                                     int* __restrict__ out_info,
                                                     int64_t n12_stride, int64_t gwork_stride,
                                                     int grp) {
  // workgroup b solves problem b of a batch: n12 n12_stride doubles apart,
  // a12g nE apart, a1r/a2r nR*d apart, scratch gwork_stride apart, one cost
  // and two info words each
  {
    const int64_t b = blockIdx.x;
    const int64_t nE_ = (int64_t)nD * nD * d * d, nRd = (int64_t)nD * D * d;
    n12 += b * n12_stride;
    a12g += b * nE_;
    a1r += b * nRd;
    a2r += b * nRd;
    gwork += b * gwork_stride;
    out_cost += b;
    out_info += 2 * b;
  }
  extern __shared__ double lds[];
  __shared__ int flag;
  __shared__ double s_d1, s_d2;
  __shared__ int s_stop;
  const int tid = threadIdx.x;
  const int nR = nD * D, d2 = d * d, nE = nD * nD * d2;
  AlsShared sh;
  sh.R = lds;
  sh.S = sh.R + (size_t)nR * nR;
  sh.a1 = sh.S + (size_t)nR * d;
  sh.a2 = sh.a1 + (size_t)nR * d;
  sh.T = sh.a2 + (size_t)nR * d;
  sh.n12g = sh.T + (size_t)grp * nD * nD * D * d;
  sh.a12n = sh.n12g + nE;
  sh.red = sh.a12n + nE;
  for (int e = tid; e < nR * d; e += ALS_NT) { sh.a1[e] = a1r[e]; sh.a2[e] = a2r[e]; }
  // n12g[Y][X][p][q] = sum_{y,x} n12[y][x][Y][X] a12g[y][x][p][q]
  als_apply_norm(n12, a12g, nD, d2, [&](int e, double v) { sh.n12g[e] = v; });
  __syncthreads();
  const double c0 = als_cost(sh, n12, nD, D, d);
  if (tid == 0) { s_d1 = fabs(c0); s_d2 = c0; s_stop = 0; }
  __syncthreads();
  int sweeps = 0, info = 0;
  for (int i = 0; i < niter; ++i) {
#pragma unroll 1
    for (int side = 0; side < 2; ++side) {
      double* own = side == 0 ? sh.a1 : sh.a2;
      als_build(sh, n12, side, nD, D, d, grp, side == 0 ? sh.a2 : sh.a1);
      if constexpr (RC == 0) als_pinv_solve(sh, nR, d, eps, gwork);
      else info |= als_solve_system<RC>(sh, nR, d, eps, &flag);
      for (int e = tid; e < nR * d; e += ALS_NT) own[e] = sh.S[e];
      __syncthreads();
    }
    sweeps = i + 1;
    const double c = als_cost(sh, n12, nD, D, d);
    if (tid == 0) {
      s_d2 = c;
      const double err = fabs(c - s_d1) / fabs(s_d1);
      s_stop = (err < tol && i > 1) ? 1 : 0;
      if (!s_stop) s_d1 = c;
    }
    __syncthreads();
    if (s_stop) break;
  }
  for (int e = tid; e < nR * d; e += ALS_NT) { a1r[e] = sh.a1[e]; a2r[e] = sh.a2[e]; }
  if (tid == 0) {
    out_cost[0] = s_d2;
    out_info[0] = sweeps;
    out_info[1] = info;
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// host wrappers
// ---------------------------------------------------------------------------
void permute_copy(const double* in, double* out, const PermDesc& p, double scale, hipStream_t s) {
  if (p.total <= 0) return;
  const int blocks = (int)std::min<int64_t>((p.total + 255) / 256, 2048);
  hipLaunchKernelGGL(permute_kernel, dim3(blocks), dim3(256), 0, s, in, out, p, scale);
  ACETN_HIP_CHECK(hipGetLastError());
}

void householder_qr(const double* A, int m, int n, double* W, double* Q, double* R,
                    hipStream_t s) {
  ACETN_REQUIRE(m >= 1 && n >= 1 && n <= kQrMaxN, "householder_qr: unsupported shape");
  hipLaunchKernelGGL(householder_qr_kernel, dim3(1), dim3(QR_NT), 0, s, A, m, n, W, Q, R);
  ACETN_HIP_CHECK(hipGetLastError());
}

namespace {
template <int NC, int R, int NWV>
void launch_qr(const QrProblem& a, const QrProblem& b, int count, int m, int n, hipStream_t s) {
  hipLaunchKernelGGL((qr_reg_kernel<NC, R, NWV>), dim3(count), dim3(64 * NWV), 0, s, a, b, m, n);
  ACETN_HIP_CHECK(hipGetLastError());
}
template <int NC, int R>
bool launch_qr_rows(const QrProblem& a, const QrProblem& b, int count, int m, int n, hipStream_t s) {
  if (m <= 64 * R) launch_qr<NC, R, 1>(a, b, count, m, n, s);
  else if (m <= 128 * R) launch_qr<NC, R, 2>(a, b, count, m, n, s);
  else if (m <= 256 * R) launch_qr<NC, R, 4>(a, b, count, m, n, s);
  else if (m <= 512 * R) launch_qr<NC, R, 8>(a, b, count, m, n, s);
  else return false;
  return true;
}
}  // namespace

void householder_qr_pair(const QrProblem& a, const QrProblem& b, int count, int m, int n,
                         double* M, double* W, hipStream_t s) {
  ACETN_REQUIRE(m >= 1 && n >= 1 && n <= kQrMaxN, "householder_qr: unsupported shape");
  // rows per thread so that the matrix and Q fit the registers
  bool done = false;
  if (n <= 4) done = launch_qr_rows<4, 4>(a, b, count, m, n, s);
  else if (n <= 8) done = launch_qr_rows<8, 4>(a, b, count, m, n, s);
  else if (n <= 12) done = launch_qr_rows<12, 4>(a, b, count, m, n, s);
  else if (n <= 16) done = launch_qr_rows<16, 2>(a, b, count, m, n, s);
  if (done) return;
  for (int i = 0; i < count; ++i) {
    const QrProblem& p = i ? b : a;
    PermDesc d{};
    d.n = 5; d.total = (int64_t)m * n;
    d.od[0] = m / (p.rd0 * p.rd1); d.od[1] = p.rd0; d.od[2] = p.rd1; d.od[3] = n / p.cd; d.od[4] = p.cd;
    for (int x = 0; x < 3; ++x) d.is[x] = p.rs[x];
    d.is[3] = p.cs[0]; d.is[4] = p.cs[1];
    permute_copy(p.A, M, d, 1.0, s);
    householder_qr(M, m, n, W, p.Q, p.R, s);
  }
}

namespace {
int svd_threads(int n) { return 64 * ((n + 3) / 4); }
}  // namespace

void svd_small(const double* A, int n, double* U, double* sv, double* V, hipStream_t s) {
  ACETN_REQUIRE(n >= 1 && n <= kSvdMaxN, "svd_small: unsupported shape");
  hipLaunchKernelGGL(svd_small_kernel, dim3(1), dim3(svd_threads(n)), 0, s, A, n, U, sv, V,
                     (int64_t)0);
  ACETN_HIP_CHECK(hipGetLastError());
}

void svd_small_batch(const double* A, int n, double* U, double* sv, double* V, int count,
                     int64_t stride, hipStream_t s) {
  ACETN_REQUIRE(n >= 1 && n <= kSvdMaxN, "svd_small: unsupported shape");
  ACETN_REQUIRE(count >= 1 && stride >= (int64_t)n * n, "svd_small_batch: bad batch layout");
  hipLaunchKernelGGL(svd_small_kernel, dim3(count), dim3(svd_threads(n)), 0, s, A, n, U, sv, V,
                     stride);
  ACETN_HIP_CHECK(hipGetLastError());
}

void lower_to_full(double* M, int n, hipStream_t s) {
  const int blocks = std::min((n * n + 255) / 256, 1024);
  hipLaunchKernelGGL(lower_to_full_kernel, dim3(blocks), dim3(256), 0, s, M, n);
  ACETN_HIP_CHECK(hipGetLastError());
}

void add_diag(double* M, int n, double shift, hipStream_t s) {
  hipLaunchKernelGGL(add_diag_kernel, dim3((n + 255) / 256), dim3(256), 0, s, M, n, shift);
  ACETN_HIP_CHECK(hipGetLastError());
}

void scale_sqrt_columns(const double* Z, const double* w, int rows, int cols, double* X,
                        hipStream_t s) {
  const int blocks = std::min((rows * cols + 255) / 256, 1024);
  hipLaunchKernelGGL(scale_sqrt_kernel, dim3(blocks), dim3(256), 0, s, Z, w, rows, cols, X);
  ACETN_HIP_CHECK(hipGetLastError());
}

void pinv_finish(const double* U, const double* sv, const double* V, int m, int n, double atol,
                 double* P, hipStream_t s) {
  hipLaunchKernelGGL(pinv_finish_kernel, dim3((n * m + 255) / 256), dim3(256), 0, s, U, sv, V, m,
                     n, atol, P);
  ACETN_HIP_CHECK(hipGetLastError());
}

void finalize_scale(const double* U, const double* sv, const double* V, int n, int bD,
                    double* r1n, double* r2n, hipStream_t s) {
  hipLaunchKernelGGL(finalize_scale_kernel, dim3(1), dim3(256), 0, s, U, sv, V, n, bD, r1n, r2n);
  ACETN_HIP_CHECK(hipGetLastError());
}

void bond_gauge(double* a1r, double* a2r, int nD1, int nD2, int bD, int pD, hipStream_t s) {
  hipLaunchKernelGGL(bond_gauge_kernel, dim3(bD), dim3(256), 0, s, a1r, a2r, nD1, nD2, bD, pD);
  ACETN_HIP_CHECK(hipGetLastError());
}

void lambda_scale(const double* A, double* out, const LambdaLegs& w, int D, int d, int invert,
                  double cutoff, hipStream_t s) {
  const int64_t n = (int64_t)D * D * D * D * d;
  const int blocks = (int)std::min<int64_t>((n + 255) / 256, 1024);
  hipLaunchKernelGGL(lambda_scale_kernel, dim3(blocks), dim3(256), 0, s, A, out, w, D, d, invert,
                     cutoff);
  ACETN_HIP_CHECK(hipGetLastError());
}

void su_split(const double* U, const double* S, const double* V, int nD, int bD, int pD,
              double* a1r, double* a2r, double* lt, hipStream_t s) {
  hipLaunchKernelGGL(su_split_kernel, dim3(1), dim3(256), 0, s, U, S, V, nD, bD, pD, a1r, a2r, lt);
  ACETN_HIP_CHECK(hipGetLastError());
}

size_t als_lds_bytes(int nD, int D, int d) {
  const size_t nR = (size_t)nD * D;
  const size_t nE = (size_t)nD * nD * d * d;
  return sizeof(double) * (nR * nR + 3 * nR * d + (size_t)nD * nD * D * d + 2 * nE + ALS_NT / 64);
}

size_t als_work_elems(int nD, int D, int d) {
  const size_t nR = (size_t)nD * D;
  return nR * nR + nR * d;
}

void als_check_shape(int nD, int D, int d, int method) {
  ACETN_REQUIRE(method == 0 || method == 1, "als: unknown method");
  ACETN_REQUIRE(method == 0 || nD * D <= 256, "als: pinv needs nD * D <= 256");
  ACETN_REQUIRE(als_lds_bytes(nD, D, d) <= 150 * 1024,
                "als: reduced tensors too large for one workgroup");
}

void als_solve_device(const double* n12, const double* a12g, double* a1r, double* a2r, int nD,
                      int D, int d, int niter, double tol, double eps, double* gwork,
                      double* out_cost, int* out_info, hipStream_t s, int method, int count) {
  ACETN_REQUIRE(count >= 1, "als: empty batch");
  als_check_shape(nD, D, d, method);
  // one problem has the CU to itself: T takes what LDS is left
  const size_t one = als_lds_bytes(nD, D, d), t1 = sizeof(double) * (size_t)nD * nD * D * d;
  const int grp = count > 1 ? 1 : (int)std::min<size_t>(nD, 1 + (150 * 1024 - one) / t1);
  const size_t lds = one + (grp - 1) * t1;
  const int64_t n12_stride = (int64_t)nD * nD * nD * nD;
  auto launch = [&](auto rc) {
    constexpr int RC = decltype(rc)::value;
    static bool attr = false;
    if (!attr) {
      ACETN_HIP_CHECK(hipFuncSetAttribute((const void*)als_kernel<RC>,
                                          hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024));
      attr = true;
    }
    hipLaunchKernelGGL(als_kernel<RC>, dim3(count), dim3(ALS_NT), lds, s, n12, a12g, a1r, a2r, nD, D, d,
                       niter, tol, eps, gwork, out_cost, out_info, n12_stride,
                       (int64_t)als_work_elems(nD, D, d), grp);
    ACETN_HIP_CHECK(hipGetLastError());
  };
  const int tiles = (nD * D + 15) / 16;
  if (method == 1) launch(std::integral_constant<int, 0>{});
  else if (tiles <= 1) launch(std::integral_constant<int, 1>{});
  else if (tiles <= 2) launch(std::integral_constant<int, 2>{});
  else if (tiles <= 3) launch(std::integral_constant<int, 3>{});
  else if (tiles <= 5) launch(std::integral_constant<int, 5>{});
  else launch(std::integral_constant<int, kAlsMaxTiles>{});
}

}  // namespace acetn
