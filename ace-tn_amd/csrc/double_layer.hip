// Double-layer absorption of one site tensor A and its conjugate into a
// block tensor X, block by block over the two outer (boundary) indices:
//
//   Y[o1,o2; k3,b3,k4,b4] = sum_{k1,b1,k2,b2,p} X[o1,o2; k1,b1,k2,b2]
//                             * A[k1,k2,k3,k4,p] * conj(A)[b1,b2,b3,b4,p]
//
// This is the pair of einsums "cuUelL,LURDP->cuelRDP" + "lurdp,cuelRDp->crRedD"
// of make_quarter_tensor (acetn/renormalization/projectors.py:54-55) and the
// pair "LURDP,alLuUx->RDPalux" + "lurdp,RDpalux->rdRDax" of renormalize_ej
// (acetn/renormalization/directional_mover.py:363-364).
//
// For a fixed boundary pair the work is two (D^2 x D^2 x D^2) products per
// physical index p:  T = X . Abar_p  and  Y += A_p^T . T, both on the matrix
// cores, in two kernels: one stacks NB blocks so that the row count is a multiple
// of the 16-row MFMA tile (NB = 4 at D = 6 gives exactly 144 rows) and works from
// LDS, the other gives each wave a block and chains the products in registers.
// Y stays in registers across p; the 7-index chi^2 D^4 d intermediate never
// reaches HBM, X and Y are read and written once.
#include "internal.h"

namespace acetn {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

// Compute type of the double-layer products: FP64 (v_mfma_f64_16x16x4f64)
// or FP32 (v_mfma_f32_16x16x4f32, the mixed-precision path).  Operands of
// both: A(16x4) lane l holds A[l%16][l/16], B(4x16) lane l holds
// B[l/16][l%16].  Results: the FP64 16x16 tile holds D[l/16 + 4r][l%16] in
// element r of lane l, the FP32 one D[4(l/16) + r][l%16].
template <typename T> struct DLMath;
template <> struct DLMath<double> {
  typedef d4 acc_t;
  static __device__ __forceinline__ acc_t mfma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return (lane >> 4) + 4 * r; }
  // result tile -> the operands of the next product's four k steps
  static __device__ __forceinline__ void to_operand(acc_t&) {}
};
template <> struct DLMath<float> {
  typedef f4 acc_t;
  static __device__ __forceinline__ acc_t mfma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
  // the 4 x 4 transpose of registers and rows of 16 lanes
  static __device__ __forceinline__ void to_operand(acc_t& z) {
    const auto swap = [](float a, float b, bool half, float& lo, float& hi) {
      const unsigned x = __float_as_uint(a), y = __float_as_uint(b);
      const auto w = half ? __builtin_amdgcn_permlane32_swap(x, y, false, false)
                          : __builtin_amdgcn_permlane16_swap(x, y, false, false);
      lo = __uint_as_float(w[0]);
      hi = __uint_as_float(w[1]);
    };
    float a, b, c, e, t0, t1, t2, t3;
    swap(z[0], z[2], true, a, c);
    swap(z[1], z[3], true, b, e);
    swap(a, b, false, t0, t1);
    swap(c, e, false, t2, t3);
    z = acc_t{t0, t1, t2, t3};
  }
};

namespace {
// 8 waves per workgroup: the LDS footprint (A, the stacked X tile and the
// intermediate T) allows one workgroup per CU at D = 6, so the waves of that
// one workgroup are what hides latency.
constexpr int NT = 512;
constexpr int NW = NT / 64;

template <int D>
struct DLShape {
  static constexpr int D2 = D * D;
  static constexpr int NB = (D == 6) ? 4 : (D == 5) ? 2 : 1;
  static constexpr int ROWS = NB * D2;            // stacked rows
  static constexpr int MP = (ROWS + 15) / 16 * 16; // padded rows (step c M, step d N)
  static constexpr int KP = (D2 + 3) / 4 * 4;      // padded contraction length
  static constexpr int XLD = KP + 1;               // odd LDS row stride of the X tile (no bank conflicts)
  static constexpr int NP = (D2 + 15) / 16 * 16;   // padded (b3,b4) columns / step d rows
  static constexpr int TC = (MP / 16) * (NP / 16); // tiles per product
  static constexpr int TPW = (TC + NW - 1) / NW;   // tiles per wave
  static constexpr int XPT = (MP * KP + NT - 1) / NT; // X elements per thread
};

template <int D>
__global__ __launch_bounds__(NT) void dl_mfma_kernel(DLDesc g, const double* __restrict__ X,
                                                     const double* __restrict__ A,
                                                     double* __restrict__ Y) {
  using S = DLShape<D>;
  using T = double;
  using M = DLMath<T>;
  typedef typename M::acc_t acc_t;
  extern __shared__ __align__(16) char smem[];
  T* sm = reinterpret_cast<T*>(smem);
  const int d = g.d;
  T* Ac = sm;                               // [p][KP][NP]: A[(l1,l2),(l3,l4),p], zero padded
  T* Xs = Ac + (size_t)d * S::KP * S::NP;   // [MP][XLD]: stacked blocks, rows (blk,k1,k2)
  T* Ts = Xs + S::MP * S::XLD;              // [MP][NP]: rows (blk,k1,k2), cols (b3,b4)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  for (int e = tid; e < d * S::KP * S::NP; e += NT) {
    const int p = e / (S::KP * S::NP), r = e % (S::KP * S::NP);
    const int kk = r / S::NP, nn = r % S::NP;
    double v = 0.0;
    if (kk < S::D2 && nn < S::D2) {
      const int l1 = kk / D, l2 = kk % D, l3 = nn / D, l4 = nn % D;
      v = A[l1 * g.a_leg[0] + l2 * g.a_leg[1] + l3 * g.a_leg[2] + l4 * g.a_leg[3] + p * g.a_p];
    }
    Ac[e] = v;
  }

  const int nblk = g.n1 * g.n2;
  const int ngroups = (nblk + S::NB - 1) / S::NB;
  // X tile of a group, element e = (row, col) of the stacked [MP][KP] tile;
  // loaded into registers one group ahead of its use.  The in-block part of
  // each element's offset is fixed, only the block base changes per group.
  T xr[S::XPT];
  int x_loff[S::XPT];
  int x_blk[S::XPT];
#pragma unroll
  for (int t = 0; t < S::XPT; ++t) {
    const int e = tid + t * NT;
    const int row = e / S::KP, col = e % S::KP;
    const int blk = row / S::D2, kk = row % S::D2;
    const bool ok = e < S::MP * S::KP && row < S::ROWS && col < S::D2;
    const int k1 = kk / D, k2 = kk % D, b1 = col / D, b2 = col % D;
    x_loff[t] = ok ? (int)(k1 * g.x_k1 + b1 * g.x_b1 + k2 * g.x_k2 + b2 * g.x_b2) : 0;
    x_blk[t] = ok ? blk : -1;
  }
  auto load_x = [&](int grp) {
    const int b0 = grp * S::NB;
    int64_t base[S::NB];
#pragma unroll
    for (int bb = 0; bb < S::NB; ++bb) {
      const int b = b0 + bb;
      base[bb] = (b < nblk) ? (int64_t)(b / g.n2) * g.x_o1 + (int64_t)(b % g.n2) * g.x_o2 : -1;
    }
#pragma unroll
    for (int t = 0; t < S::XPT; ++t) {
      int64_t bo = -1;
#pragma unroll
      for (int bb = 0; bb < S::NB; ++bb)
        if (x_blk[t] == bb) bo = base[bb];
      xr[t] = bo < 0 ? 0.0 : X[bo + x_loff[t]];
    }
  };
  if ((int)blockIdx.x < ngroups) load_x(blockIdx.x);
  for (int grp = blockIdx.x; grp < ngroups; grp += gridDim.x) {
    const int b0 = grp * S::NB;
    __syncthreads();
    // ---- stacked X tile (from registers), then start loading the next group
#pragma unroll
    for (int t = 0; t < S::XPT; ++t) {
      const int e = tid + t * NT;
      if (e < S::MP * S::KP) Xs[(e / S::KP) * S::XLD + e % S::KP] = xr[t];
    }
    if (grp + (int)gridDim.x < ngroups) load_x(grp + gridDim.x);
    acc_t yacc[S::TPW];
#pragma unroll
    for (int t = 0; t < S::TPW; ++t) yacc[t] = acc_t{0, 0, 0, 0};

    // closed: sum_p A_p^T (X Abar_p);  open: every (p, pb) pair written out
    for (int pb = 0; pb < d; ++pb) {
      const T* Apb = Ac + (size_t)pb * S::KP * S::NP;
      __syncthreads();
      // ---- step c: Ts[MP x NP] = Xs[MP x KP] . Abar_pb[KP x NP]
#pragma unroll
      for (int t = 0; t < S::TPW; ++t) {
        const int tile = t * NW + wave;  // round-robin over the waves (even SIMD load)
        if (tile < S::TC) {
          const int tm = tile / (S::NP / 16), tn = tile % (S::NP / 16);
          acc_t acc = acc_t{0, 0, 0, 0};
#pragma unroll 3
          for (int ks = 0; ks < S::KP; ks += 4) {
            const T a = Xs[(tm * 16 + (lane & 15)) * S::XLD + ks + (lane >> 4)];
            const T b = Apb[(ks + (lane >> 4)) * S::NP + tn * 16 + (lane & 15)];
            acc = M::mfma(a, b, acc);
          }
          for (int r = 0; r < 4; ++r)
            Ts[(tm * 16 + M::row(lane, r)) * S::NP + tn * 16 + (lane & 15)] = acc[r];
        }
      }
      __syncthreads();
      const int p_lo = g.open_p ? 0 : pb, p_hi = g.open_p ? d : pb + 1;
      for (int p = p_lo; p < p_hi; ++p) {
        const T* Ap = Ac + (size_t)p * S::KP * S::NP;
        if (g.open_p) {
#pragma unroll
          for (int t = 0; t < S::TPW; ++t) yacc[t] = acc_t{0, 0, 0, 0};
        }
        // ---- step d: Y[(k3,k4), (blk,b3,b4)] += A_p^T[(k3,k4),(k1,k2)] . T[(blk,k1,k2),(b3,b4)]
#pragma unroll
        for (int t = 0; t < S::TPW; ++t) {
          const int tile = t * NW + wave;  // round-robin over the waves (even SIMD load)
          if (tile < S::TC) {
            const int tm = tile / (S::MP / 16), tn = tile % (S::MP / 16);
            const int nn = tn * 16 + (lane & 15);
            const int blk = nn / S::D2, b34 = nn % S::D2;
#pragma unroll 3
            for (int ks = 0; ks < S::KP; ks += 4) {
              const int kk = ks + (lane >> 4);
              const T a = Ap[kk * S::NP + tm * 16 + (lane & 15)];
              const T b = (kk < S::D2 && nn < S::ROWS) ? Ts[(blk * S::D2 + kk) * S::NP + b34] : T(0);
              yacc[t] = M::mfma(a, b, yacc[t]);
            }
          }
        }
        if (g.open_p || (p == d - 1)) {
          const int64_t poff = g.open_p ? (int64_t)p * g.y_p + (int64_t)pb * g.y_pb : 0;
          // ---- write Y (after the last p when closed, per (p, pb) when open)
#pragma unroll
          for (int t = 0; t < S::TPW; ++t) {
            const int tile = t * NW + wave;  // round-robin over the waves (even SIMD load)
            if (tile < S::TC) {
              const int tm = tile / (S::MP / 16), tn = tile % (S::MP / 16);
              const int nn = tn * 16 + (lane & 15);
              const int blk = nn / S::D2, b34 = nn % S::D2;
              if (nn < S::ROWS && b0 + blk < nblk) {
                const int o1 = (b0 + blk) / g.n2, o2 = (b0 + blk) % g.n2;
                const int64_t yb = (int64_t)o1 * g.y_o1 + (int64_t)o2 * g.y_o2 + poff;
                const int b3 = b34 / D, b4 = b34 % D;
                for (int r = 0; r < 4; ++r) {
                  const int m = tm * 16 + M::row(lane, r);
                  if (m < S::D2) {
                    const int k3 = m / D, k4 = m % D;
                    const int64_t yo = yb + k3 * g.y_k3 + b3 * g.y_b3 + k4 * g.y_k4 + b4 * g.y_b4;
                    Y[yo] = yacc[t][r];
                  }
                }
              }
            }
          }
        }
      }
    }
  }
}

// The same two products, a boundary block a wave: X is read straight into the
// operands of the first (rows (k1,k2), k (b1,b2)), whose result tiles are the
// second's operands, so a wave meets no barrier and only A is in LDS.  One column
// tile of (b3,b4) at a time, X kept for all of them.  More padding than the
// stacked rows above at D = 5 and 6, no intermediate in LDS; bound by the
// scattered loads and stores (32 - 48 byte pieces) and, in FP64, by the products.
// The order of sums is that of the stacked kernel, bit for bit.
template <int D, typename T>
__global__ __launch_bounds__(256) void dl_wave_kernel(DLDesc g, const double* __restrict__ X,
                                                      const double* __restrict__ A,
                                                      double* __restrict__ Y) {
  using M = DLMath<T>;
  typedef typename M::acc_t acc_t;
  constexpr int D2 = D * D, NT = (D2 + 15) / 16, KS = (D2 + 3) / 4, KP = 4 * KS, NP = 16 * NT;
  extern __shared__ __align__(16) char smem[];
  int64_t* yrow = reinterpret_cast<int64_t*>(smem);  // (k3, k4)
  int64_t* ycol = yrow + NP;                         // (b3, b4)
  T* Ac = reinterpret_cast<T*>(ycol + NP);           // [p][KP][NP], zero padded
  const int d = g.d;
  const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, kq = lane >> 4;
  for (int e = tid; e < d * KP * NP; e += 256) {
    const int p = e / (KP * NP), r = e % (KP * NP), kk = r / NP, nn = r % NP;
    double v = 0.0;
    if (kk < D2 && nn < D2)
      v = A[kk / D * g.a_leg[0] + kk % D * g.a_leg[1] + nn / D * g.a_leg[2] + nn % D * g.a_leg[3] +
            p * g.a_p];
    Ac[e] = (T)v;
  }
  if (tid < NP) {
    const int i = min(tid, D2 - 1);
    yrow[tid] = i / D * g.y_k3 + i % D * g.y_k4;
    ycol[tid] = i / D * g.y_b3 + i % D * g.y_b4;
  }
  __syncthreads();
  int xrow[NT], xcol[KS];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int i = min(16 * t + m, D2 - 1);
    xrow[t] = (int)(i / D * g.x_k1 + i % D * g.x_k2);
  }
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int i = min(4 * s + kq, D2 - 1);
    xcol[s] = (int)(i / D * g.x_b1 + i % D * g.x_b2);
  }
  const int nblk = g.n1 * g.n2, nwave = gridDim.x * 4;
  for (int blk = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(tid >> 6); blk < nblk;
       blk += nwave) {
    const int o1 = blk / g.n2, o2 = blk % g.n2;
    const int64_t xo = o1 * g.x_o1 + o2 * g.x_o2, yo = o1 * g.y_o1 + o2 * g.y_o2;
    T xa[NT][KS];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int64_t at = xo + xrow[t] + xcol[s];
        const T v = g.x_f32 ? (T)reinterpret_cast<const float*>(X)[at] : (T)X[at];
        // padding rows and columns hold zeros where a product reaches them
        const bool ok = (KP == D2 || 4 * s + kq < D2) && (KP == D2 || 16 * t + m < D2);
        xa[t][s] = ok ? v : T(0);
      }
#pragma unroll 1
    for (int tn = 0; tn < NT; ++tn) {
      acc_t y[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) y[t] = acc_t{0, 0, 0, 0};
      // closed: sum_p A_p^T (X Abar_p);  open: every (p, pb) pair written out
#pragma unroll 1
      for (int pb = 0; pb < d; ++pb) {
        const T* Ab = Ac + (size_t)pb * KP * NP + kq * NP + tn * 16 + m;
        acc_t z[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) z[t] = acc_t{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const T b = Ab[4 * s * NP];
#pragma unroll
          for (int t = 0; t < NT; ++t) z[t] = M::mfma(xa[t][s], b, z[t]);
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) M::to_operand(z[t]);
        const int p_hi = g.open_p ? d : pb + 1;
#pragma unroll 1
        for (int p = g.open_p ? 0 : pb; p < p_hi; ++p) {
          const T* Ap = Ac + (size_t)p * KP * NP + kq * NP + m;
          if (g.open_p) {
#pragma unroll
            for (int t = 0; t < NT; ++t) y[t] = acc_t{0, 0, 0, 0};
          }
#pragma unroll
          for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int t = 0; t < NT; ++t)
              y[t] = M::mfma(Ap[4 * s * NP + 16 * t], z[s >> 2][s & 3], y[t]);
          if (!g.open_p && p < d - 1) continue;
          const int64_t yc = yo + ycol[16 * tn + m] +
                             (g.open_p ? p * g.y_p + pb * g.y_pb : (int64_t)0);
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int row = 16 * t + M::row(lane, r);
              if (16 * tn + m >= D2 || row >= D2) continue;
              const int64_t at = yc + yrow[row];
              if (g.y_f32) reinterpret_cast<float*>(Y)[at] = (float)y[t][r];
              else Y[at] = (double)y[t][r];
            }
        }
      }
    }
  }
}

// one round of resident workgroups, each looping over its share of the blocks:
// the A tensor is staged once per workgroup
template <int D>
void launch_dl_stacked(const DLDesc& g, const double* X, const double* A, double* Y, hipStream_t s) {
  using S = DLShape<D>;
  static_assert(S::TC == (S::NP / 16) * (S::MP / 16), "tile counts of the two products differ");
  const size_t lds = sizeof(double) * ((size_t)g.d * S::KP * S::NP + (size_t)S::MP * S::XLD +
                                       (size_t)S::MP * S::NP);
  ACETN_REQUIRE(lds <= 160 * 1024, "double_layer: LDS budget exceeded");
  static bool attr = false;
  if (!attr) {
    ACETN_HIP_CHECK(hipFuncSetAttribute((const void*)dl_mfma_kernel<D>,
                                        hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    attr = true;
  }
  const int64_t ngroups = ((int64_t)g.n1 * g.n2 + S::NB - 1) / S::NB;
  const int per_cu = (int)std::max<size_t>(1, std::min<size_t>(8, (160 * 1024) / lds));
  const int grid = (int)std::min<int64_t>(ngroups, 256 * per_cu);
  hipLaunchKernelGGL(dl_mfma_kernel<D>, dim3(grid), dim3(NT), lds, s, g, X, A, Y);
}

template <int D, typename T>
void launch_dl_wave(const DLDesc& g, const double* X, const double* A, double* Y, hipStream_t s) {
  constexpr int NP = (D * D + 15) / 16 * 16, KP = (D * D + 3) / 4 * 4;
  constexpr int kPerCu = D >= 5 && sizeof(T) == 8 ? 3 : 4;  // D=6: 256, 247, 293 us at 2, 3, 4
  const size_t lds = 16 * NP + sizeof(T) * (size_t)g.d * KP * NP;
  static bool attr = false;
  if (!attr) {
    ACETN_HIP_CHECK(hipFuncSetAttribute((const void*)dl_wave_kernel<D, T>,
                                        hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    attr = true;
  }
  const int per_cu = (int)std::max<size_t>(1, std::min<size_t>(kPerCu, (160 * 1024) / lds));
  const int grid = (int)std::min<int64_t>(((int64_t)g.n1 * g.n2 + 3) / 4, 256 * per_cu);
  hipLaunchKernelGGL((dl_wave_kernel<D, T>), dim3(grid), dim3(256), lds, s, g, X, A, Y);
}

// Which kernel: the wave one wherever it was the faster (us, stacked / wave;
// FP32 D=6 198 / 164, D=8 2890 / 2730; FP64 D=2 6.5 / 3.6, D=3 6.0 / 4.5, D=4
// 10.1 / 8, D=5 82 / 72, D=6 258 / 247), the stacked one for FP64 at D = 7 and 8
// (385 / 398, 452 / 487) and, from D = 5, with the physical legs open (D=5 144 /
// 166: four times the stores).
template <int D, typename T>
void launch_dl(const DLDesc& g, const double* X, const double* A, double* Y, hipStream_t s) {
  ACETN_REQUIRE((int64_t)(D - 1) * (g.x_k1 + g.x_b1 + g.x_k2 + g.x_b2) < (int64_t(1) << 31),
                "double_layer: block strides exceed 32-bit offsets");
  const double d2 = (double)D * D, d6 = d2 * d2 * d2, nblk = (double)g.n1 * g.n2;
  const double flops = nblk * (2.0 * g.d * d6 + 2.0 * (g.open_p ? g.d * g.d : g.d) * d6);
  hipEvent_t e0 = kernel_timing_begin(s);
  if constexpr (sizeof(T) == 8 && D >= 5) {
    if (D > 6 || g.open_p) launch_dl_stacked<D>(g, X, A, Y, s);
    else launch_dl_wave<D, T>(g, X, A, Y, s);
  } else {
    launch_dl_wave<D, T>(g, X, A, Y, s);
  }
  ACETN_HIP_CHECK(hipGetLastError());
  // algorithmic bytes: the X blocks read once, the Y blocks written once
  const double yblk = g.open_p ? (double)g.d * g.d : 1.0;
  const double xb = g.x_f32 ? 4.0 : 8.0, yb = g.y_f32 ? 4.0 : 8.0;
  kernel_timing_end(e0, s, kKDoubleLayer, flops, nblk * d2 * d2 * (xb + yb * yblk));
}

template <typename T>
void double_layer_t(const DLDesc& g, const double* X, const double* A, double* Y, hipStream_t s) {
  ACETN_REQUIRE(g.d >= 1 && g.d <= 4, "double_layer: d must be in [1, 4]");
  if ((int64_t)g.n1 * g.n2 <= 0) return;
  switch (g.D) {
    case 1: launch_dl<1, T>(g, X, A, Y, s); break;
    case 2: launch_dl<2, T>(g, X, A, Y, s); break;
    case 3: launch_dl<3, T>(g, X, A, Y, s); break;
    case 4: launch_dl<4, T>(g, X, A, Y, s); break;
    case 5: launch_dl<5, T>(g, X, A, Y, s); break;
    case 6: launch_dl<6, T>(g, X, A, Y, s); break;
    case 7: launch_dl<7, T>(g, X, A, Y, s); break;
    case 8: launch_dl<8, T>(g, X, A, Y, s); break;
    default: ACETN_REQUIRE(false, "double_layer: D must be in [1, 8]");
  }
}
}  // namespace

void double_layer_f64(const DLDesc& g, const double* X, const double* A, double* Y,
                      hipStream_t s) {
  ACETN_REQUIRE(!g.x_f32 && !g.y_f32, "double_layer_f64: FP64 X and Y only");
  double_layer_t<double>(g, X, A, Y, s);
}

void double_layer_f32(const DLDesc& g, const double* X, const double* A, double* Y,
                      hipStream_t s) {
  double_layer_t<float>(g, X, A, Y, s);
}

// ---------------------------------------------------------------------------
// The closing contraction of a one-site network,
//
//   Y[r,u; l,b,p] = sum_{e,R,c,U} T3[e; r,R; c; u,U] sum_{L,B} T1[c; l,L; e; b,B]
//                                 * conj(A)[L,U,R,B,p]
//
// (T1 c4.e4.e3, T3 the other three sides).  Block (c, e) of the boundary gives
// two D^2 x D^2 x D^2 products per p, Z = A_p^T T1 and Y_p += T3 Z, chained in
// registers: an element r of the 16 x 16 result tile tm of Z is the operand of
// k step 4 tm + r.  Wave (p, tn) of a workgroup keeps column tile tn of Y_p over
// all its blocks; the workgroups' sums are added in a fixed order.  As two
// products over memory, with the chi^2 D^4 d intermediate between them, D=5,
// chi=100 took 470 us; so 55 us, bound by the loads of the two tensors
// (100 MB, 48 - 200 bytes at a stretch).
// ---------------------------------------------------------------------------
namespace {
constexpr int kRingWGs = 512;
constexpr int kRingP = 2;  // physical indices a launch: 8 waves at most, 256 registers

template <int D>
__global__ __launch_bounds__(64 * kRingP * ((D * D + 15) / 16)) void ring_close_kernel(
    const double* __restrict__ T1, const double* __restrict__ T3, const double* __restrict__ A,
    int ne, int nc, int d, int p0, double* __restrict__ part) {
  constexpr int D2 = D * D, NT = (D2 + 15) / 16, KS = (D2 + 3) / 4;
  extern __shared__ __align__(16) double Ac[];  // [p][k = (L, B)][row = (R, U)], zero padded
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, m = lane & 15, kq = lane >> 4;
  const int np = (int)blockDim.x / (64 * NT);  // indices p0 .. p0 + np - 1 of d
  for (int x = tid; x < np * KS * 4 * NT * 16; x += blockDim.x) {
    const int row = x % (NT * 16), k = x / (NT * 16) % (KS * 4), p = p0 + x / (NT * 16 * KS * 4);
    double v = 0.0;
    if (row < D2 && k < D2) {
      const int L = k / D, B = k % D, R = row / D, U = row % D;
      v = A[((((int64_t)L * D + U) * D + R) * D + B) * d + p];
    }
    Ac[x] = v;
  }
  __syncthreads();
  const int p = wave / NT, tn = wave % NT;
  const double* Ap = Ac + (size_t)p * KS * 4 * NT * 16;
  const int64_t s1 = (int64_t)ne * D2, s3 = (int64_t)nc * D2;
  // this lane's column (l, b) of T1 and rows (r, u) of T3
  const int cl = min(tn * 16 + m, D2 - 1);
  const int64_t c1 = (int64_t)(cl / D) * D * s1 + cl % D * D;
  d4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = d4{0.0, 0.0, 0.0, 0.0};
  for (int blk = blockIdx.x; blk < ne * nc; blk += gridDim.x) {
    const int c = blk / ne, e = blk % ne;
    const double* x1 = T1 + c * (int64_t)D2 * s1 + (int64_t)e * D2 + c1;
    double xb[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int k = 4 * ks + kq, kc = min(k, D2 - 1);
      const double v = x1[kc / D * s1 + kc % D];
      xb[ks] = k < D2 ? v : 0.0;
    }
    d4 z[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      z[t] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        z[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(Ap[(4 * ks + kq) * NT * 16 + t * 16 + m],
                                                    xb[ks], z[t], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if constexpr (NT > 3) __builtin_amdgcn_sched_barrier(0);  // one row tile's loads at a time
      const int rw = min(t * 16 + m, D2 - 1);
      const double* x3 = T3 + ((int64_t)e * D + rw / D) * D * s3 + (int64_t)c * D2 + rw % D * D;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int k = 4 * ks + kq, kc = min(k, D2 - 1);
        const double v = x3[kc / D * s3 + kc % D];
        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(k < D2 ? v : 0.0, z[ks >> 2][ks & 3], acc[t],
                                                      0, 0, 0);
      }
    }
  }
  double* out = part + (int64_t)blockIdx.x * D2 * D2 * d + p0 + p;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = t * 16 + kq + 4 * r, col = tn * 16 + m;
      if (row < D2 && col < D2) out[((int64_t)row * D2 + col) * d] = acc[t][r];
    }
}

// Y = the sum of the workgroups' parts: 16 elements a workgroup, 16 threads
// each summing every 16th part, then those in order
__global__ __launch_bounds__(256) void ring_sum_kernel(const double* __restrict__ part, int n,
                                                       int parts, double* __restrict__ Y) {
  __shared__ double red[16][16];
  const int o = threadIdx.x & 15, g = threadIdx.x >> 4, e = blockIdx.x * 16 + o;
  double s = 0.0;
  if (e < n) {
#pragma unroll 8
    for (int w = g; w < parts; w += 16) s += part[(int64_t)w * n + e];
  }
  red[g][o] = s;
  __syncthreads();
  if (g > 0 || e >= n) return;
  for (int w = 1; w < 16; ++w) s += red[w][o];
  Y[e] = s;
}

template <int D>
void launch_ring(const double* T1, const double* T3, const double* A, int ne, int nc, int d,
                 double* part, int wgs, hipStream_t s) {
  constexpr int D2 = D * D, NT = (D2 + 15) / 16, KS = (D2 + 3) / 4;
  for (int p0 = 0; p0 < d; p0 += kRingP) {
    const int np = std::min(kRingP, d - p0);
    const size_t lds = sizeof(double) * (size_t)np * KS * 4 * NT * 16;  // 64 KB at D = 8
    hipLaunchKernelGGL(ring_close_kernel<D>, dim3(wgs), dim3(64 * np * NT), lds, s, T1, T3, A, ne,
                       nc, d, p0, part);
  }
}
}  // namespace

size_t ring_close_work_elems(int D, int d, int ne, int nc) {
  return (size_t)std::min<int64_t>(kRingWGs, (int64_t)ne * nc) * D * D * D * D * d;
}

void ring_close(const double* T1, const double* T3, const double* A, int D, int d, int ne, int nc,
                double* work, double* Y, hipStream_t s) {
  ACETN_REQUIRE(D >= 1 && D <= 8 && d >= 1 && ne >= 1 && nc >= 1 &&
                    (int64_t)ne * nc < (int64_t(1) << 31),
                "ring_close: unsupported shape");
  const int wgs = (int)std::min<int64_t>(kRingWGs, (int64_t)ne * nc), n = D * D * D * D * d;
  switch (D) {
    case 1: launch_ring<1>(T1, T3, A, ne, nc, d, work, wgs, s); break;
    case 2: launch_ring<2>(T1, T3, A, ne, nc, d, work, wgs, s); break;
    case 3: launch_ring<3>(T1, T3, A, ne, nc, d, work, wgs, s); break;
    case 4: launch_ring<4>(T1, T3, A, ne, nc, d, work, wgs, s); break;
    case 5: launch_ring<5>(T1, T3, A, ne, nc, d, work, wgs, s); break;
    case 6: launch_ring<6>(T1, T3, A, ne, nc, d, work, wgs, s); break;
    case 7: launch_ring<7>(T1, T3, A, ne, nc, d, work, wgs, s); break;
    default: launch_ring<8>(T1, T3, A, ne, nc, d, work, wgs, s); break;
  }
  ACETN_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(ring_sum_kernel, dim3((n + 15) / 16), dim3(256), 0, s, work, n, wgs, Y);
  ACETN_HIP_CHECK(hipGetLastError());
}

}  // namespace acetn
