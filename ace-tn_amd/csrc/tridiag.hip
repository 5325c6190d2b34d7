// Approximate eigenvectors of a symmetric FP64 matrix (32 < q <= kTridiagMaxQ) through its
// tridiagonal form: what the projector SVD is preconditioned with.
//   * Householder tridiagonalisation, one workgroup: the whole matrix in
//     registers up to q = 192, read from L2 in panels above;
//   * one wave per eigenpair, all over the chip: its eigenvalue by 64-way
//     multisection on the Sturm count, its vector by two steps of inverse
//     iteration from a random start, and the Householder reflectors applied to
//     it in registers.
// The vectors satisfy G x = w x to about eps |G|.  Those of a cluster of
// eigenvalues span its invariant subspace but, coming from independent random
// starts, are not orthogonal: the caller orthonormalises the set (it is well
// conditioned: vectors of separate eigenvalues are orthogonal to eps |G| / gap,
// and those of one cluster are random in its subspace).
#include "internal.h"
#include "lanes.h"

#include <cmath>

namespace acetn {
namespace {

// The reflector H = I - tau u u^T that takes a column with leading entry alpha
// and |rest|^2 = s2 to beta e_1: u = (alpha - beta, rest).  False: nothing to
// do (the rest vanishes, or is negligible next to a matrix of norm one).
__device__ __forceinline__ bool reflector(double alpha, double s2, double& beta, double& u0,
                                          double& tau) {
  beta = alpha;
  u0 = 0.0;
  tau = 0.0;
  if (!(s2 > 1e-280)) return false;
  const double x = fma(alpha, alpha, s2);
  beta = -copysign(x * rsqrt_nr(x), alpha);
  u0 = alpha - beta;
  tau = -rcp_nr(beta * u0);
  return true;
}

// 1 / (largest |diagonal entry|), the scale that brings a positive
// semidefinite matrix to norm of order one (1 when it vanishes).
__device__ __forceinline__ double diag_scale(const double* G, int q, int lane) {
  double dm = 0.0;
  for (int i = lane; i < q; i += 64) dm = fmax(dm, fabs(G[(int64_t)i * q + i]));
  for (int o = 32; o > 0; o >>= 1) dm = fmax(dm, __shfl_xor(dm, o));
  return (dm > 1e-290 && dm < 1e290) ? 1.0 / dm : 1.0;
}

// --------------------------------------------------------------------------
// q <= 32 NB: thread (ty, tx) of a 32 x 16 grid holds the entries
// (ty + 32 A, tx + 16 B).  A step costs two barriers: the 16 lanes that hold
// row k (= column k) make the reflector u from their registers and publish it,
// then the product p = A u is published.  Everything a wave would repeat for
// itself counts four-fold (the waves share four SIMDs), so eight waves with
// more entries each beat sixteen, and only the owners compute the reflector.
// The rank-2 update and p skip the 32-blocks that are already reduced; rows
// and columns that are done with go on being rotated, which changes no norm
// and is never read.
// U: row k holds reflector k (zeros up to k), tau[k] its factor.
// --------------------------------------------------------------------------
constexpr int TR_NT = 512;
constexpr int kTrRegMaxQ = 192;

template <int NB>
__global__ __launch_bounds__(TR_NT) void tridiag_reg_kernel(const double* __restrict__ G, int q,
                                                            double* __restrict__ U,
                                                            double* __restrict__ tau,
                                                            double* __restrict__ d,
                                                            double* __restrict__ e) {
  __shared__ double su[2][32 * NB], sp[32 * NB], st[2];
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  const double sc = diag_scale(G, q, tid & 63);
  double a[NB][2 * NB];
#pragma unroll
  for (int A = 0; A < NB; ++A)
#pragma unroll
    for (int B = 0; B < 2 * NB; ++B) {
      const int i = ty + 32 * A, j = tx + 16 * B;
      const int lo = min(i, j), hi = max(i, j);
      a[A][B] = hi < q ? sc * G[(int64_t)lo * q + hi] : 0.0;
    }
#pragma unroll
  for (int K = 0; K < NB; ++K) {
    for (int kk = 0; kk < 32; ++kk) {
      const int k = 32 * K + kk;
      if (k >= q) break;
      double* su_ = su[k & 1];
      if (ty == kk) {
        double s2 = 0.0, alpha = 0.0;
#pragma unroll
        for (int B = 2 * K; B < 2 * NB; ++B) {
          const int j = tx + 16 * B;
          const double v = a[K][B];
          if (j > k + 1) s2 = fma(v, v, s2);
          if (j == k + 1) alpha = v;
          if (j == k) d[k] = v;
        }
        s2 = sum16(s2);
        alpha = sum16(alpha);
        double beta, u0, t;
        reflector(alpha, s2, beta, u0, t);
#pragma unroll
        for (int B = 0; B < 2 * NB; ++B) {
          const int j = tx + 16 * B;
          const double v = (B < 2 * K || t == 0.0 || j <= k) ? 0.0 : (j == k + 1 ? u0 : a[K][B]);
          if (B >= 2 * K) su_[j] = v;
          if (j < q) U[(int64_t)k * q + j] = v;
        }
        if (tx == 0) {
          st[k & 1] = t;
          tau[k] = t;
          e[k] = beta;
        }
      }
      __syncthreads();
      const double t = st[k & 1];
      double uc[2 * NB];
      if (t != 0.0) {
#pragma unroll
        for (int B = 2 * K; B < 2 * NB; ++B) uc[B] = su_[tx + 16 * B];
#pragma unroll
        for (int A = K; A < NB; ++A) {
          double s = 0.0;
#pragma unroll
          for (int B = 2 * K; B < 2 * NB; ++B) s = fma(a[A][B], uc[B], s);
          s = sum16(s);
          if (tx == A) sp[ty + 32 * A] = s;
        }
      }
      __syncthreads();
      if (t != 0.0) {
        double wc[2 * NB], g = 0.0;
#pragma unroll
        for (int B = 2 * K; B < 2 * NB; ++B) {
          wc[B] = sp[tx + 16 * B];
          g = fma(uc[B], wc[B], g);
        }
        g = 0.5 * t * sum16(g);
#pragma unroll
        for (int B = 2 * K; B < 2 * NB; ++B) wc[B] = t * fma(-g, uc[B], wc[B]);
#pragma unroll
        for (int A = K; A < NB; ++A) {
          const double ur = su_[ty + 32 * A];
          const double wr = t * fma(-g, ur, sp[ty + 32 * A]);
#pragma unroll
          for (int B = 2 * K; B < 2 * NB; ++B)
            a[A][B] = fma(-wr, uc[B], fma(-ur, wc[B], a[A][B]));
        }
      }
    }
  }
}

// --------------------------------------------------------------------------
// kTrRegMaxQ < q <= kTridiagMaxQ: the matrix is kept in global memory (it stays in L2)
// and updated once per panel of 16 reflectors, on the matrix cores; a step
// reads the trailing matrix once for p = A u, every wave its share of rows
// with the columns spread over its lanes, and corrects for the panel's own
// reflectors (V, W in LDS).  Bound by that read from one CU (about 64 B a
// clock).
// --------------------------------------------------------------------------
constexpr int kTgNB = 16;
constexpr int kTgR = (kTridiagMaxQ + 63) / 64;  // columns per lane
constexpr int TG_NW = 16;
typedef double tr_d4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(64 * TG_NW) void tridiag_glb_kernel(
    const double* __restrict__ G, int q, double* __restrict__ S, double* __restrict__ U,
    double* __restrict__ tau, double* __restrict__ d, double* __restrict__ e) {
  // dynamic LDS: V, W (kTgNB x ld each), the rows' partial products
  // (TG_NW / 2 x ld, two waves each), u
  extern __shared__ double sm[];
  const int ld = (q + 15) / 16 * 16;
  double* V = sm;
  double* W = V + kTgNB * ld;
  double* part = W + kTgNB * ld;
  double* u = part + TG_NW / 2 * ld;
  __shared__ double red[TG_NW], dots[2 * kTgNB];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int NT = 64 * TG_NW;
  const double sc = diag_scale(G, q, lane);
  // S: ld x ld, zero padding
  for (int x = tid; x < ld * ld; x += NT) {
    const int i = x / ld, j = x % ld;
    const int lo = min(i, j), hi = max(i, j);
    S[x] = hi < q ? sc * G[(int64_t)lo * q + hi] : 0.0;
  }
  __syncthreads();
  auto block_sum = [&](double x) {
    x = sum64(x);
    if (lane == 0) red[wave] = x;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < TG_NW; ++w) s += red[w];
    return s;
  };
  for (int p0 = 0; p0 < q; p0 += kTgNB) {
    const int nb = min(kTgNB, q - p0);
    for (int x = tid; x < 2 * kTgNB * ld; x += NT) sm[x] = 0.0;
    __syncthreads();
    for (int t = 0; t < nb; ++t) {
      const int k = p0 + t;
      // column k of the current matrix (thread j: entry j >= k)
      double c = 0.0;
      if (tid < q && tid >= k) {
        c = S[(int64_t)k * ld + tid];
        for (int r = 0; r < t; ++r)
          c -= V[r * ld + k] * W[r * ld + tid] + W[r * ld + k] * V[r * ld + tid];
      }
      if (tid == k) d[k] = c;
      if (tid < ld) u[tid] = tid > k ? c : 0.0;
      const double s2 = block_sum(tid > k + 1 && tid < q ? c * c : 0.0);
      if (k + 1 >= q) break;
      double beta, u0, ta;
      const bool on = reflector(u[k + 1], s2, beta, u0, ta);
      __syncthreads();
      if (tid == 0) {
        e[k] = beta;
        tau[k] = ta;
        u[k + 1] = u0;
      }
      __syncthreads();
      if (tid < q) U[(int64_t)k * q + tid] = on ? u[tid] : 0.0;
      if (!on) continue;  // V and W of this step stay zero
      // p = A u: wave w takes rows k + 1 + w, ..., lane l columns l, l + 64, ...
      double acc[kTgR];
#pragma unroll
      for (int r = 0; r < kTgR; ++r) acc[r] = 0.0;
      const int r0 = (k + 1) >> 6;  // column blocks below are done with
      // four rows at a time: the loads of all of them in flight together
      for (int i = k + 1 + wave; i < q; i += 4 * TG_NW) {
        double ui[4], v[4][kTgR];
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const int ix = min(i + x * TG_NW, ld - 1);
          ui[x] = i + x * TG_NW < q ? u[ix] : 0.0;
          const double* row = S + (int64_t)ix * ld + lane;
#pragma unroll
          for (int r = 0; r < kTgR; ++r)
            v[x][r] = (r >= r0 && 64 * r + lane < ld) ? row[64 * r] : 0.0;
        }
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
          for (int r = 0; r < kTgR; ++r) acc[r] = fma(ui[x], v[x][r], acc[r]);
      }
      // the panel's corrections need W^T u and V^T u
      for (int x = wave; x < 2 * t; x += TG_NW) {
        const double* P = (x & 1 ? V : W) + (x >> 1) * ld;
        double s = 0.0;
        for (int j = lane; j < q; j += 64) s = fma(P[j], u[j], s);
        s = sum64(s);
        if (lane == 0) dots[x] = s;
      }
      // sum the waves' partials: the upper half of the waves hands over first
      if (wave >= TG_NW / 2) {
#pragma unroll
        for (int r = 0; r < kTgR; ++r)
          if (64 * r + lane < ld) part[(wave - TG_NW / 2) * ld + 64 * r + lane] = acc[r];
      }
      __syncthreads();
      if (wave < TG_NW / 2) {
#pragma unroll
        for (int r = 0; r < kTgR; ++r)
          if (64 * r + lane < ld) part[wave * ld + 64 * r + lane] += acc[r];
      }
      __syncthreads();
      double pj = 0.0;
      if (tid < q && tid > k) {
#pragma unroll
        for (int w = 0; w < TG_NW / 2; ++w) pj += part[w * ld + tid];
        for (int r = 0; r < t; ++r)
          pj -= V[r * ld + tid] * dots[2 * r] + W[r * ld + tid] * dots[2 * r + 1];
      }
      const double uj = tid < ld ? u[tid] : 0.0;
      const double g = 0.5 * ta * block_sum(pj * uj);
      if (tid < q && tid > k) {
        V[t * ld + tid] = uj;
        W[t * ld + tid] = ta * (pj - g * uj);
      }
      __syncthreads();
    }
    if (p0 + kTgNB >= q) break;
    __syncthreads();
    // S -= V^T W + W^T V on the trailing tiles, one 16 x 16 tile per wave
    const int T0 = p0 / 16 + 1, nt = ld / 16 - T0;
    const int m = lane & 15, kq = lane >> 4;
    for (int x = wave; x < nt * nt; x += TG_NW) {
      const int I = 16 * (T0 + x / nt), J = 16 * (T0 + x % nt);
      tr_d4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = S[(int64_t)(I + kq + 4 * r) * ld + J + m];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const int t = 4 * ks + kq;
        v = __builtin_amdgcn_mfma_f64_16x16x4f64(-V[t * ld + I + m], W[t * ld + J + m], v, 0, 0, 0);
        v = __builtin_amdgcn_mfma_f64_16x16x4f64(-W[t * ld + I + m], V[t * ld + J + m], v, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) S[(int64_t)(I + kq + 4 * r) * ld + J + m] = v[r];
    }
    __syncthreads();
  }
}

// --------------------------------------------------------------------------
// Eigenpair j (descending) of the tridiagonal matrix, one wave per workgroup,
// written as row j of X after the back-transformation.  The recurrences are
// serial in the matrix index: the multisection runs 64 of them side by side
// (one shift a lane), the factorisation and solves of the inverse iteration
// run once, the same in every lane.  Latency-bound: about 9 counts, a
// factorisation and 2 solves of q dependent steps, then q reflectors; operands
// come from LDS eight steps at a time, ahead of the chain that uses them.
// Padding up to a multiple of eight: diagonal entries far above the spectrum,
// not coupled, which add no eigenvalue below any shift and solve to zero.
// --------------------------------------------------------------------------
// uniform in (-1, 1): an xorshift-multiply mix of both numbers, with two prime
// multipliers of xxHash and the rounds of Wellons' hash-prospector [15 2c1b3c6d
// 12 297a2d39 15]
__device__ __forceinline__ double hash_uniform(unsigned a, unsigned b) {
  unsigned h = a * 0x9E3779B1u ^ (b + 0x7F4A7C15u) * 0x85EBCA77u;
  h ^= h >> 15; h *= 0x2C1B3C6Du;
  h ^= h >> 12; h *= 0x297A2D39u;
  h ^= h >> 15;
  return ((double)h + 0.5) * (2.0 / 4294967296.0) - 1.0;
}

template <int R>
__global__ __launch_bounds__(64) void tri_vectors_kernel(const double* __restrict__ d,
                                                         const double* __restrict__ e,
                                                         const double* __restrict__ U,
                                                         const double* __restrict__ tau, int q,
                                                         double* __restrict__ X,
                                                         double* __restrict__ lam) {
  constexpr int MQ = 64 * R;
  __shared__ __align__(16) double sd[MQ + 8], se[MQ + 8], se2[MQ + 8];
  __shared__ __align__(16) double iD[MQ + 8], U1[MQ + 8], U2[MQ + 8], L[MQ + 8], x[MQ + 8];
  __shared__ unsigned char piv[MQ / 8 + 1];
  const int lane = threadIdx.x, j = blockIdx.x;
  const int q8 = (q + 7) / 8 * 8;
  // Gershgorin interval
  double lo = INFINITY, hi = -INFINITY;
  for (int i = lane; i < q; i += 64) {
    const double di = d[i], er = i + 1 < q ? e[i] : 0.0, el = i > 0 ? e[i - 1] : 0.0;
    const double r = fabs(er) + fabs(el);
    lo = fmin(lo, di - r);
    hi = fmax(hi, di + r);
  }
  for (int o = 32; o > 0; o >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, o));
    hi = fmax(hi, __shfl_xor(hi, o));
  }
  const double nrm = fmax(fabs(lo), fabs(hi));
  const double tiny = fmax(nrm * 2.2e-16, 1e-290);
  lo -= 4.0 * tiny;
  hi += 4.0 * tiny;
  for (int i = lane; i < q8; i += 64) {
    const double er = i + 1 < q ? e[i] : 0.0, el = (i > 0 && i < q) ? e[i - 1] : 0.0;
    sd[i] = i < q ? d[i] : 3.0 * nrm + 1.0;
    se[i] = er;
    // never quite zero, so that a minor that vanishes next to a vanishing
    // coupling does not end the sequence
    se2[i] = fmax(el * el, 1e-50);
  }
  __syncthreads();
  // multisection: the number of eigenvalues below s from the signs of the
  // principal minors p_i = (d_i - s) p_{i-1} - e_{i-1}^2 p_{i-2}, rescaled
  // every 8 steps (the matrix has norm of order one, so 8 steps stay in range)
  const int below = q - 1 - j;  // eigenvalues below the wanted one
  for (int round = 0; round < 10 && hi - lo > tiny; ++round) {
    const double w = (hi - lo) / 65.0;
    const double s = lo + w * (lane + 1);
    double pm = 0.0, pc = 1.0;  // p_{i-2}, p_{i-1}
    int count = 0;
    for (int i0 = 0; i0 < q8; i0 += 8) {
      double dd[8], ee[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        dd[i] = sd[i0 + i] - s;
        ee[i] = se2[i0 + i];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const double pn = fma(dd[i], pc, -ee[i] * pm);
        count += (__double2hiint(pn) ^ __double2hiint(pc)) < 0;
        pm = pc;
        pc = pn;
      }
      const int ex = max(__builtin_amdgcn_frexp_exp(pm), __builtin_amdgcn_frexp_exp(pc));
      pm = ldexp(pm, -ex);
      pc = ldexp(pc, -ex);
    }
    const unsigned long long above = __ballot(count > below);
    const int f = above ? __ffsll(above) - 1 : 64;
    const double nlo = f > 0 ? lo + w * f : lo;
    const double nhi = f < 64 ? lo + w * (f + 1) : hi;
    lo = nlo;
    hi = nhi;
  }
  const double s = 0.5 * (lo + hi);
  if (lane == 0) lam[j] = s;
  // T - s = P L U with partial pivoting (the same in every lane)
  {
    double dc = sd[0] - s, uc = se[0];
    for (int i0 = 0; i0 < q8; i0 += 8) {
      double cc[8], dn[8], un[8], r0[8], r1[8], r2[8], r3[8];
      unsigned pb = 0;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        cc[i] = se[i0 + i];
        dn[i] = (i0 + i + 1 < q8 ? sd[i0 + i + 1] : 1.0) - s;
        un[i] = i0 + i + 1 < q8 ? se[i0 + i + 1] : 0.0;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const double c = cc[i];
        const bool sw = fabs(c) > fabs(dc);
        double top = sw ? c : dc;
        top = fabs(top) < tiny ? copysign(tiny, top) : top;
        const double inv = rcp_nr(top), mlt = (sw ? dc : c) * inv;
        r0[i] = inv;
        r1[i] = sw ? dn[i] : uc;
        r2[i] = sw ? un[i] : 0.0;
        r3[i] = mlt;
        pb |= sw ? 1u << i : 0u;
        dc = fma(-mlt, r1[i], sw ? uc : dn[i]);
        uc = sw ? -mlt * un[i] : un[i];
      }
      if (lane == 0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          iD[i0 + i] = r0[i];
          U1[i0 + i] = r1[i];
          U2[i0 + i] = r2[i];
          L[i0 + i] = r3[i];
        }
        piv[i0 / 8] = (unsigned char)pb;
      }
    }
  }
  for (int i = lane; i < q8; i += 64)
    x[i] = i < q ? hash_uniform((unsigned)j, (unsigned)i) : 0.0;
  __syncthreads();
  double v[R];
  for (int it = 0; it < 2; ++it) {
    {
      double b = x[0];
      for (int i0 = 0; i0 < q8; i0 += 8) {
        double bn[8], l[8], o[8];
        const unsigned pb = piv[i0 / 8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          bn[i] = i0 + i + 1 < q8 ? x[i0 + i + 1] : 0.0;
          l[i] = L[i0 + i];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const bool sw = (pb >> i) & 1;
          o[i] = sw ? bn[i] : b;
          b = fma(-l[i], o[i], sw ? b : bn[i]);
        }
        if (lane == 0) {
#pragma unroll
          for (int i = 0; i < 8; ++i) x[i0 + i] = o[i];
        }
      }
    }
    __syncthreads();
    {
      double x1 = 0.0, x2 = 0.0;
      for (int i0 = q8 - 8; i0 >= 0; i0 -= 8) {
        double b[8], u1[8], u2[8], r[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          r[i] = iD[i0 + i];
          b[i] = x[i0 + i] * r[i];
          u1[i] = U1[i0 + i] * r[i];
          u2[i] = U2[i0 + i] * r[i];
        }
#pragma unroll
        for (int i = 7; i >= 0; --i) {
          const double xi = fma(-u1[i], x1, fma(-u2[i], x2, b[i]));
          x2 = x1;
          x1 = xi;
          b[i] = xi;
        }
        if (lane == 0) {
#pragma unroll
          for (int i = 0; i < 8; ++i) x[i0 + i] = b[i];
        }
      }
    }
    __syncthreads();
    double mx = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      v[r] = lane + 64 * r < q ? x[lane + 64 * r] : 0.0;
      mx = fmax(mx, fabs(v[r]));
    }
    for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o));
    const double sc = 1.0 / mx;
    double n2 = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      v[r] *= sc;
      n2 = fma(v[r], v[r], n2);
    }
    const double inv = 1.0 / sqrt(sum64(n2));
#pragma unroll
    for (int r = 0; r < R; ++r) {
      v[r] *= inv;
      if (it == 0 && lane + 64 * r < q) x[lane + 64 * r] = v[r];
    }
    __syncthreads();
  }
  // back-transformation: v <- H_0 H_1 ... H_{q-2} v, two reflectors loaded
  // while two are applied
  double un[2][R], tn[2];
  auto load = [&](int k) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int kh = max(k - h, 0);
      tn[h] = k - h >= 0 ? tau[kh] : 0.0;
#pragma unroll
      for (int r = 0; r < R; ++r)
        un[h][r] = lane + 64 * r < q ? U[(int64_t)kh * q + lane + 64 * r] : 0.0;
    }
  };
  if (q >= 2) load(q - 2);
  for (int k = q - 2; k >= 0; k -= 2) {
    double u[2][R], t[2], g0 = 0.0, g1 = 0.0, h = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      u[0][r] = un[0][r];
      u[1][r] = un[1][r];
      g0 = fma(u[0][r], v[r], g0);
      g1 = fma(u[1][r], v[r], g1);
      h = fma(u[0][r], u[1][r], h);
    }
    t[0] = tn[0];
    t[1] = tn[1];
    if (k >= 2) load(k - 2);
    // H_{k-1} H_k v = v - g0 u0 - g1' u1, g1' = t1 u1.(v - g0 u0)
    g0 = t[0] * sum64(g0);
    g1 = t[1] * fma(-g0, sum64(h), sum64(g1));
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = fma(-g1, u[1][r], fma(-g0, u[0][r], v[r]));
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (lane + 64 * r < q) X[(int64_t)j * q + lane + 64 * r] = v[r];
}

// --------------------------------------------------------------------------
// One step of the iterative refinement of a symmetric eigen-decomposition
// (Ogita and Aishima, Japan J. Indust. Appl. Math. 35, 2018): for a basis X
// with S = X^T G X and H = X^T X close to diagonal and to I, X (I + E) has
// both errors squared, with
//   l_i = S_ii / H_ii,  E_ij = (S_ij - l_j H_ij) / (l_j - l_i),  E_ii = (1 - H_ii) / 2.
// Pairs whose E_ij is not small (close or equal eigenvalues, or noise next to
// negligible ones) are left to the Jacobi solve that follows: E_ij = -H_ij / 2
// only keeps them orthonormal.  The test weighs E_ij by sqrt(l_i / l_j) where
// that is larger, its share in the smaller of the two singular directions.
// A step leaves the basis orthonormal to its largest E_ij squared, so the
// limit falls from the first step (most, 1e-4) to the last (1e-8): what the
// last step finds between close values is rounding noise over their gap.
// F = I when the basis was judged not to be worth it.
// --------------------------------------------------------------------------
constexpr int RF_ROWS = 4;

__global__ __launch_bounds__(256) void refine_kernel(const double* __restrict__ S,
                                                     const double* __restrict__ H, int q,
                                                     double* __restrict__ F,
                                                     const int* __restrict__ robust,
                                                     double most) {
  __shared__ double l[512];
  for (int i = threadIdx.x; i < q; i += 256)
    l[i] = S[(int64_t)i * q + i] / H[(int64_t)i * q + i];
  const bool skip = *robust != 0;
  __syncthreads();
  const int i0 = blockIdx.x * RF_ROWS;
  for (int x = threadIdx.x; x < RF_ROWS * q; x += 256) {
    const int i = i0 + x / q, j = x % q;
    if (i >= q) break;
    const double li = l[i], lj = l[j];
    // both triangles: E_ij + E_ji = -H_ij is what keeps the basis orthonormal,
    // so S and H enter symmetrised and a pair is taken or left as a whole
    const double h = 0.5 * (H[(int64_t)i * q + j] + H[(int64_t)j * q + i]);
    const double sij = 0.5 * (S[(int64_t)i * q + j] + S[(int64_t)j * q + i]);
    double f;
    if (skip) {
      f = i == j ? 1.0 : 0.0;
    } else if (i == j) {
      f = 1.0 + 0.5 * (1.0 - h);
    } else {
      const double m2 = most * most, inv = 1.0 / (lj - li);
      f = (sij - lj * h) * inv;
      const double g = (li * h - sij) * inv, f2 = f * f, g2 = g * g;  // E_ij, E_ji
      const bool ok = f2 <= m2 && g2 <= m2 && f2 * li <= m2 * lj && g2 * lj <= m2 * li;
      if (!ok) f = -0.5 * h;
    }
    F[(int64_t)i * q + j] = f;
  }
}

// Whether the tridiagonal route serves this matrix (one workgroup).  Not when
//   * the spectrum is graded: singular values below 1e-4 of the largest.
//     Jacobi rotations of a graded matrix keep the small components of its
//     vectors to relative accuracy, a tridiagonal form only to eps |G|: the
//     projector column of s_j is then good to eps s_0 / s_j, 1e-12 at this line;
//   * four or more eigenvalues agree to the accuracy of the tridiagonal form:
//     inverse iteration weighs the directions of so large a cluster by rounding
//     noise, and its vectors come out too close to dependent;
//   * the orthonormalised basis is off by more than the two refinement steps
//     square away (or is not finite).
constexpr double kGraded = 1e-8, kCluster = 3e-14, kBasisOff = 1e-4;

__global__ __launch_bounds__(1024) void judge_kernel(const double* __restrict__ lam,
                                                     const double* __restrict__ H, int q,
                                                     int* __restrict__ robust) {
  const double l0 = lam[0];
  int bad = !(l0 > 0.0 && lam[q - 1] >= kGraded * l0);
  for (int j = threadIdx.x; j + 3 < q; j += 1024) bad |= !(lam[j] - lam[j + 3] >= kCluster * l0);
  for (int x = threadIdx.x; x < q * q; x += 1024)
    bad |= !(fabs(H[x] - (x / q == x % q ? 1.0 : 0.0)) <= kBasisOff);
  bad = __syncthreads_or(bad);
  if (threadIdx.x == 0) *robust = bad ? 1 : 0;
}

size_t tridiag_ld(int q) { return (size_t)(q + 15) / 16 * 16; }

}  // namespace

size_t tridiag_scratch_elems(int q) {
  // reflectors, tau, d, e and the working copy of the global variant
  const size_t ld = tridiag_ld(q);
  return (size_t)q * q + 3 * (size_t)q + (q > kTrRegMaxQ ? ld * ld : 0);
}

void tridiag_vectors(const double* G, double* X, double* lam, int q, double* scratch,
                     hipStream_t s) {
  ACETN_REQUIRE(q > 32 && q <= kTridiagMaxQ, "tridiag_vectors: q out of range");
  double* U = scratch;
  double* tau = U + (size_t)q * q;
  double* d = tau + q;
  double* e = d + q;
  if (q <= kTrRegMaxQ) {
#define ACETN_TR(NB) \
  hipLaunchKernelGGL(tridiag_reg_kernel<NB>, dim3(1), dim3(TR_NT), 0, s, G, q, U, tau, d, e)
    switch ((q + 31) / 32) {
      case 2: ACETN_TR(2); break;
      case 3: ACETN_TR(3); break;
      case 4: ACETN_TR(4); break;
      case 5: ACETN_TR(5); break;
      default: ACETN_TR(6); break;
    }
#undef ACETN_TR
  } else {
    const size_t lds = sizeof(double) * tridiag_ld(q) * (2 * kTgNB + TG_NW / 2 + 1);
    constexpr size_t most = sizeof(double) * kTridiagMaxQ * (2 * kTgNB + TG_NW / 2 + 1);
    static_assert(kTridiagMaxQ % 16 == 0 && most <= 156 * 1024,
                  "the panel of the largest matrix has to fit the LDS");
    static bool attr = false;
    if (!attr) {
      ACETN_HIP_CHECK(hipFuncSetAttribute((const void*)tridiag_glb_kernel,
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)most));
      attr = true;
    }
    hipLaunchKernelGGL(tridiag_glb_kernel, dim3(1), dim3(64 * TG_NW), lds, s, G, q, e + q, U, tau,
                       d, e);
  }
  ACETN_HIP_CHECK(hipGetLastError());
#define ACETN_TV(R) \
  hipLaunchKernelGGL(tri_vectors_kernel<R>, dim3(q), dim3(64), 0, s, d, e, U, tau, q, X, lam)
  switch ((q + 63) / 64) {
    case 1: ACETN_TV(1); break;
    case 2: ACETN_TV(2); break;
    case 3: ACETN_TV(3); break;
    case 4: ACETN_TV(4); break;
    case 5: ACETN_TV(5); break;
    case 6: ACETN_TV(6); break;
    case 7: ACETN_TV(7); break;
    default: ACETN_TV(8); break;
  }
#undef ACETN_TV
  ACETN_HIP_CHECK(hipGetLastError());
}

void judge_basis(const double* lam, const double* H, int q, int* robust, hipStream_t s) {
  hipLaunchKernelGGL(judge_kernel, dim3(1), dim3(1024), 0, s, lam, H, q, robust);
  ACETN_HIP_CHECK(hipGetLastError());
}

void refine_eigenvectors(const double* S, const double* H, int q, double* F, const int* robust,
                         double most, hipStream_t s) {
  ACETN_REQUIRE(q >= 1 && q <= 512, "refine_eigenvectors: q out of range");
  hipLaunchKernelGGL(refine_kernel, dim3((q + RF_ROWS - 1) / RF_ROWS), dim3(256), 0, s, S, H, q, F,
                     robust, most);
  ACETN_HIP_CHECK(hipGetLastError());
}

}  // namespace acetn
