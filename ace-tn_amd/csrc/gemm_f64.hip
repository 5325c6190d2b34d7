// FP64 GEMM on the CDNA4 matrix cores (v_mfma_f64_16x16x4_f64).
//
// One kernel serves every contraction of the CTMRG / full-update path: each
// operand is addressed through two-level index maps, so the index
// permutations the reference performs with torch.einsum transposes are folded
// into the global->LDS tile loads instead of being materialised in HBM.
//
// Tiles: 4 waves in a 2 x 2 arrangement, each owning WM x WN MFMA blocks of
// 16 x 16 (workgroup tile 32*WM x 32*WN, chosen per shape), BK = 16.  Operand
// fragments follow the MFMA register layout: A(16x4) lane l holds
// A[l%16][l/16], B(4x16) lane l holds B[l/16][l%16], and the 16x16 f64
// result lane l holds D[l/16 + 4r][l%16], r = 0..3 (checked on gfx950).
// Long-K / few-tile problems are split along K into a deterministic partial
// buffer that a second kernel reduces (no atomics, bitwise reproducible).
#include "internal.h"

#include <mutex>
#include <vector>

namespace acetn {

typedef double d4 __attribute__((ext_vector_type(4)));

// ---- optional live timing of the matrix-core kernel launches (HIP events on
// the launch stream), per kernel class, used by the benchmark for the
// roofline figures.
namespace {
struct KTimer {
  std::mutex mu;
  bool on = false;
  struct Rec { hipEvent_t e0, e1; int cls; };
  std::vector<Rec> ev;
  double flops[kKClasses] = {};
  double bytes[kKClasses] = {};
  int64_t launches[kKClasses] = {};
};
KTimer& ktimer() {
  static KTimer t;
  return t;
}
}  // namespace

void kernel_timing_enable(bool on) {
  KTimer& t = ktimer();
  std::lock_guard<std::mutex> g(t.mu);
  for (auto& e : t.ev) { (void)hipEventDestroy(e.e0); (void)hipEventDestroy(e.e1); }
  t.ev.clear();
  for (int c = 0; c < kKClasses; ++c) { t.flops[c] = 0.0; t.bytes[c] = 0.0; t.launches[c] = 0; }
  t.on = on;
}

void kernel_timing_read(int cls, double* ms, double* flops, int64_t* launches) {
  ACETN_REQUIRE(cls >= 0 && cls < kKClasses, "kernel_timing_read: unknown kernel class");
  KTimer& t = ktimer();
  std::lock_guard<std::mutex> g(t.mu);
  double tot = 0.0;
  for (auto& e : t.ev) {
    if (e.cls != cls) continue;
    ACETN_HIP_CHECK(hipEventSynchronize(e.e1));
    float x = 0.f;
    ACETN_HIP_CHECK(hipEventElapsedTime(&x, e.e0, e.e1));
    tot += x;
  }
  *ms = tot;
  *flops = t.flops[cls];
  *launches = t.launches[cls];
}

hipEvent_t kernel_timing_begin(hipStream_t s) {
  KTimer& t = ktimer();
  if (!t.on) return nullptr;
  hipEvent_t e0 = nullptr;
  ACETN_HIP_CHECK(hipEventCreate(&e0));
  ACETN_HIP_CHECK(hipEventRecord(e0, s));
  return e0;
}

double kernel_timing_bytes(int cls) {
  ACETN_REQUIRE(cls >= 0 && cls < kKClasses, "kernel_timing_bytes: unknown kernel class");
  KTimer& t = ktimer();
  std::lock_guard<std::mutex> g(t.mu);
  return t.bytes[cls];
}

void kernel_timing_end(hipEvent_t e0, hipStream_t s, int cls, double flops, double bytes) {
  if (e0 == nullptr) return;
  KTimer& t = ktimer();
  hipEvent_t e1 = nullptr;
  ACETN_HIP_CHECK(hipEventCreate(&e1));
  ACETN_HIP_CHECK(hipEventRecord(e1, s));
  std::lock_guard<std::mutex> lg(t.mu);
  t.ev.push_back({e0, e1, cls});
  t.flops[cls] += flops;
  t.bytes[cls] += bytes;
  t.launches[cls] += 1;
}

namespace {
constexpr int BK = 16, NT = 256;

__device__ __forceinline__ bool contiguous(const IdxMap& m) { return m.s0 == 1; }

// Workgroup tile BM x BN with BM = 16*WM*WGM, BN = 32*WN: WGM x 2 waves
// (WGM = 2 or 4), each wave owning WM x WN MFMA blocks of 16 x 16, k-tiles
// of BKT (16 or 32).  Double-buffered LDS (one barrier per k-tile) with the
// next tile prefetched into registers; more waves or longer k-tiles give the
// global loads more MFMA work to hide behind.
// LIN: every operand map is a single stride (no grouped digits), so an
// element's address is base + row*stride + k*stride: rows past the edge are
// clamped to the last row (their results are never stored) and only the K
// edge needs a predicate, which keeps the tile loads free of branches.
// Otherwise the k part of the address (a mixed-radix map) is evaluated once
// per k-tile and operand by 2*BK threads into a double-buffered LDS table
// that every element load reads, instead of once per element.
// Four-wave tiles up to 2 x 5 blocks per wave are held to 256 VGPRs, so two
// workgroups share a CU (their LDS fits twice); larger tiles and the
// eight-wave variants take the registers they need.
template <int WM, int WN, bool LIN, int WGM = 2, int BKT = BK>
__global__ __launch_bounds__(128 * WGM, (WGM == 2 && WM < 4 && BKT == 16) ? 2 : 1) void
gemm_f64_kernel(GemmDesc g, GemmBatch bt, int ksplit, double* __restrict__ work) {
  constexpr int NT = 128 * WGM;
  constexpr int BK = BKT;
  constexpr int BM = 16 * WM * WGM, BN = 32 * WN;
  constexpr int LA = BM + 2, LB = BN + 2;
  constexpr int AE = BM * BK / NT, BE = BN * BK / NT;  // elements per thread
  static_assert(AE * NT == BM * BK && BE * NT == BN * BK, "tile not divisible by the threads");
  __shared__ double As[2][BK][LA];
  __shared__ double Bs[2][BK][LB];
  __shared__ int64_t koff[2][2][BK];  // [table][operand A / B][k within the tile]
  if (g.run_if && *g.run_if == 0) return;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int prob = blockIdx.z / ksplit, kpart = blockIdx.z % ksplit;
  const double* __restrict__ A = bt.A[prob];
  const double* __restrict__ B = bt.B[prob];
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;

  int kchunk = (g.K + ksplit - 1) / ksplit;
  kchunk = (kchunk + BK - 1) / BK * BK;
  const int kbeg = kpart * kchunk;
  const int kend = min(g.K, kbeg + kchunk);

  // ---- load patterns (coalesced along whichever index is unit-stride)
  const bool a_mfast = contiguous(g.am) || !contiguous(g.ak);
  int a_ml[AE], a_kl[AE];
  int64_t a_moff[AE];
  bool a_mok[AE];
#pragma unroll
  for (int i = 0; i < AE; ++i) {
    const int e = tid + i * NT;
    if (a_mfast) { a_ml[i] = e % BM; a_kl[i] = e / BM; }
    else         { a_kl[i] = e % BK; a_ml[i] = e / BK; }
    const int m = m0 + a_ml[i];
    a_mok[i] = m < g.M;
    if (LIN) a_moff[i] = (int64_t)min(m, g.M - 1) * g.am.s0;
    else a_moff[i] = a_mok[i] ? imap(g.am, m) : 0;
  }
  const bool b_nfast = contiguous(g.bn) || !contiguous(g.bk);
  int b_nl[BE], b_kl[BE];
  int64_t b_noff[BE];
  bool b_nok[BE];
#pragma unroll
  for (int i = 0; i < BE; ++i) {
    const int e = tid + i * NT;
    if (b_nfast) { b_nl[i] = e % BN; b_kl[i] = e / BN; }
    else         { b_kl[i] = e % BK; b_nl[i] = e / BK; }
    const int n = n0 + b_nl[i];
    b_nok[i] = n < g.N;
    if (LIN) b_noff[i] = (int64_t)min(n, g.N - 1) * g.bn.s0;
    else b_noff[i] = b_nok[i] ? imap(g.bn, n) : 0;
  }

  d4 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};

  double ra[AE], rb[BE];
  auto load_tile = [&](int kt) {
    if (LIN) {
      const int64_t sak = g.ak.s0, sbk = g.bk.s0;
#pragma unroll
      for (int i = 0; i < AE; ++i) {
        const int k = kt + a_kl[i];
        const double v = A[a_moff[i] + (int64_t)min(k, kend - 1) * sak];
        ra[i] = k < kend ? v : 0.0;
      }
#pragma unroll
      for (int i = 0; i < BE; ++i) {
        const int k = kt + b_kl[i];
        const double v = B[(int64_t)min(k, kend - 1) * sbk + b_noff[i]];
        rb[i] = k < kend ? v : 0.0;
      }
      return;
    }
    const int tb = ((kt - kbeg) / BK) & 1;
#pragma unroll
    for (int i = 0; i < AE; ++i) {
      const int k = kt + a_kl[i];
      ra[i] = (a_mok[i] && k < kend) ? A[a_moff[i] + koff[tb][0][a_kl[i]]] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < BE; ++i) {
      const int k = kt + b_kl[i];
      rb[i] = (b_nok[i] && k < kend) ? B[koff[tb][1][b_kl[i]] + b_noff[i]] : 0.0;
    }
  };
  // k-offset table of the k-tile at kt (general maps only)
  auto fill_koff = [&](int kt) {
    if (LIN || tid >= 2 * BK) return;
    const int tb = ((kt - kbeg) / BK) & 1, op = tid / BK, j = tid % BK;
    const int k = min(kt + j, kend - 1);
    koff[tb][op][j] = op == 0 ? imap(g.ak, k) : imap(g.bk, k);
  };
  auto store_tile = [&](int buf) {
#pragma unroll
    for (int i = 0; i < AE; ++i) As[buf][a_kl[i]][a_ml[i]] = ra[i];
#pragma unroll
    for (int i = 0; i < BE; ++i) Bs[buf][b_kl[i]][b_nl[i]] = rb[i];
  };

  int buf = 0;
  if (kbeg < kend) {
    if (!LIN) {
      fill_koff(kbeg);
      __syncthreads();
    }
    load_tile(kbeg);
    store_tile(0);
    if (kbeg + BK < kend) fill_koff(kbeg + BK);
  }
  __syncthreads();
  for (int kt = kbeg; kt < kend; kt += BK) {
    const bool more = kt + BK < kend;
    if (more) load_tile(kt + BK);  // global loads in flight during the MFMAs
#pragma unroll
    for (int ks = 0; ks < BK / 4; ++ks) {
      const int kr = ks * 4 + (lane >> 4);
      double a[WM], b[WN];
#pragma unroll
      for (int i = 0; i < WM; ++i) a[i] = As[buf][kr][wm * 16 * WM + i * 16 + (lane & 15)];
#pragma unroll
      for (int j = 0; j < WN; ++j) b[j] = Bs[buf][kr][wn * 16 * WN + j * 16 + (lane & 15)];
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    if (more) store_tile(buf ^ 1);
    // the table of k-tile kt + 2 BK replaces that of kt, read before the
    // previous barrier
    if (kt + 2 * BK < kend) fill_koff(kt + 2 * BK);
    __syncthreads();
    buf ^= 1;
  }

  // ---- epilogue
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm * 16 * WM + i * 16 + (lane >> 4) + 4 * r;
        const int n = n0 + wn * 16 * WN + j * 16 + (lane & 15);
        if (m >= g.M || n >= g.N) continue;
        const double v = acc[i][j][r];
        if (ksplit == 1) {
          double* C = bt.C[prob];
          const int64_t off = imap(g.cm, m) + imap(g.cn, n);
          C[off] = (g.beta != 0.0) ? g.alpha * v + g.beta * C[off] : g.alpha * v;
        } else {
          work[(((int64_t)prob * ksplit + kpart) * g.M + m) * g.N + n] = v;
        }
      }
}

__global__ void splitk_reduce_kernel(GemmDesc g, GemmBatch bt, int ksplit,
                                     const double* __restrict__ work) {
  if (g.run_if && *g.run_if == 0) return;
  const int64_t mn = (int64_t)g.M * g.N;
  const int prob = blockIdx.y;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < mn;
       e += (int64_t)gridDim.x * blockDim.x) {
    // eight partial loads in flight per step; the sum keeps the part order
    const double* wp = work + (int64_t)prob * ksplit * mn + e;
    double s = 0.0;
    int p = 0;
    for (; p + 8 <= ksplit; p += 8) {
      double v[8];
#pragma unroll
      for (int t = 0; t < 8; ++t) v[t] = wp[(int64_t)(p + t) * mn];
#pragma unroll
      for (int t = 0; t < 8; ++t) s += v[t];
    }
    for (; p < ksplit; ++p) s += wp[(int64_t)p * mn];
    const int m = (int)(e / g.N), n = (int)(e % g.N);
    double* C = bt.C[prob];
    const int64_t off = imap(g.cm, m) + imap(g.cn, n);
    C[off] = (g.beta != 0.0) ? g.alpha * s + g.beta * C[off] : g.alpha * s;
  }
}

// --------------------------------------------------------------------------
// Large products with plainly strided operands: A contiguous along k or along
// m (AM), B along n, all rows even and 16-byte aligned.  One workgroup of four
// waves makes a 64 x 16 WN tile, 16 rows a wave, in k-tiles of 16; two
// workgroups share a CU, so that one's barriers and stores fall into the
// other's products (one workgroup of eight waves, in step at every barrier,
// took 11 % longer; LDS and memory instructions dealt out between the matrix
// instructions 10 % longer still).
//
// At these shapes the matrix cores are the bound (64 clocks a 16x16x4 product,
// 128 flop a clock and CU), so everything else has to stay out of their way:
//   * 16-byte loads, three k-tiles ahead in two sets of registers;
//   * the operands of each product are read from LDS while the one before runs;
//   * the k index is dealt so that a lane needs neighbouring k's in two
//     successive products: 16-byte LDS reads of a k-contiguous A, whose 16-byte
//     pieces are xor-ed over the banks, and rows of A (AM) and B padded so that
//     two of the four k groups of a read cover the 64 banks;
//   * the width in steps of 16 columns: 146 columns pay for 160, 66 for 80;
//   * the number of k parts from the rounds of workgroups that result
//     (pipe_ksplit), instead of a part count that leaves a last round nearly
//     empty.
// Measured with the reduction of the parts, back to back, against the 64- and
// 128-row tiles of gemm_f64_kernel: 5184 x 146 x 5184 (the range finder at
// D=6, chi=144) 200 us against 295 (its matrix-core floor is 110 us at 72
// TFLOP/s: power holds the clock near 2.2 GHz, and the operands' way in costs
// the rest), 2500 x 102 x 2500 47 against 74, 2592 x 74 x 2592 37 against 41,
// 1024 x 66 x 1024 17 against 20.
// --------------------------------------------------------------------------
constexpr int PP_NW = 4, PP_NT = 64 * PP_NW, PP_BM = 16 * PP_NW, PP_BK = 16, PP_MAXWN = 10;
typedef double pd2 __attribute__((ext_vector_type(2)));

template <int WN, bool AM>
__global__ __launch_bounds__(PP_NT, 2) void gemm_f64_pipe_kernel(GemmDesc g, const double* __restrict__ A,
                                                                 const double* __restrict__ B,
                                                                 double* __restrict__ C, int ksplit,
                                                                 double* __restrict__ work) {
  constexpr int BN = 16 * WN, LDB = BN + 8;
  constexpr int LDA = PP_BM + 8;                        // AM: row of k
  constexpr int SA = AM ? PP_BK * LDA : PP_BM * PP_BK;  // doubles per buffer
  constexpr int SB = PP_BK * LDB;
  constexpr int NB = (8 * PP_BK * WN + PP_NT - 1) / PP_NT;  // 16-byte pieces of B per thread
  __shared__ __align__(16) double sA[2][SA];
  __shared__ __align__(16) double sB[2][SB];
  if (g.run_if && *g.run_if == 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m16 = lane & 15, kq = lane >> 4;
  const int m0 = blockIdx.y * PP_BM, n0 = blockIdx.x * BN, kpart = blockIdx.z;
  const int64_t lda = AM ? g.ak.s0 : g.am.s0, ldb = g.bk.s0;
  const int ktiles = (g.K + PP_BK - 1) / PP_BK;
  const int per = (ktiles + ksplit - 1) / ksplit;
  const int kbeg = kpart * per * PP_BK;
  const int kend = min(g.K, kbeg + per * PP_BK);
  const int nst = kend > kbeg ? (kend - kbeg + PP_BK - 1) / PP_BK : 0;

  // this thread's pieces: (row, piece) of A and (k, piece) of B; rows and
  // columns past the edge are clamped (their results are never stored)
  int ax[2], ay[2], bx[NB], by[NB];
  const double* ap[2];
  const double* bp[NB];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int x = tid + PP_NT * i;
    ax[i] = AM ? x / (PP_BM / 2) : x >> 3;  // k, or m
    ay[i] = AM ? x % (PP_BM / 2) : x & 7;   // piece of m, or of k
    ap[i] = AM ? A + (int64_t)min(m0 + 2 * ay[i], (g.M - 1) & ~1)
               : A + (int64_t)min(m0 + ax[i], g.M - 1) * lda;
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int x = min(tid + PP_NT * i, 8 * PP_BK * WN - 1);
    bx[i] = x / (8 * WN);
    by[i] = x % (8 * WN);
    bp[i] = B + min(n0 + 2 * by[i], (g.N - 1) & ~1);
  }
  struct Regs {
    pd2 a[2], b[NB];
  };
  // piece i of k-tile st: the two of A, then those of B
  constexpr int NP = 2 + NB;
  auto load = [&](int st, Regs& r, int i) {
    const int k0 = kbeg + st * PP_BK;
    if (i >= 2) {
      r.b[i - 2] = *reinterpret_cast<const pd2*>(
          bp[i - 2] + (int64_t)min(k0 + bx[i - 2], kend - 1) * ldb);
    } else if (AM) {
      const int k = k0 + ax[i];
      r.a[i] = *reinterpret_cast<const pd2*>(ap[i] + (int64_t)min(k, kend - 1) * lda);
    } else {
      r.a[i] = *reinterpret_cast<const pd2*>(ap[i] + min(k0 + 2 * ay[i], (kend - 1) & ~1));
    }
  };
  auto store = [&](int st, const Regs& r, int i) {
    if (i >= 2) {
      *reinterpret_cast<pd2*>(&sB[st & 1][bx[i - 2] * LDB + 2 * by[i - 2]]) = r.b[i - 2];
      return;
    }
    const int at = AM ? ax[i] * LDA + 2 * ay[i] : ax[i] * PP_BK + 2 * (ay[i] ^ (ax[i] & 7));
    *reinterpret_cast<pd2*>(&sA[st & 1][at]) = r.a[i];
  };
  // zeros past the last k, in both operands (what was loaded there may be
  // infinite): a branch that only a ragged last k-tile takes
  auto zero_past_end = [&](int st, Regs& r) {
    const int k0 = kbeg + st * PP_BK;
    if (k0 + PP_BK <= kend) return;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int k = k0 + (AM ? ax[i] : 2 * ay[i]);
      if (k >= kend) r.a[i].x = 0.0;
      if (AM ? k >= kend : k + 1 >= kend) r.a[i].y = 0.0;
    }
#pragma unroll
    for (int i = 0; i < NB; ++i)
      if (k0 + bx[i] >= kend) r.b[i] = pd2{0.0, 0.0};
  };
  d4 acc[WN];
#pragma unroll
  for (int j = 0; j < WN; ++j) acc[j] = d4{0.0, 0.0, 0.0, 0.0};
  // operands of the four products of a k-tile, two sets of registers in turn:
  // product x = 2 t + h takes k = 8 t + 2 kq + h
  pd2 a[2];
  double b[2][WN];
  const int row = 16 * wave + m16;
  auto fetch_a = [&](int buf, int x) {
    const int k = 8 * (x >> 1) + 2 * kq + (x & 1);
    if (AM) {
      if (x & 1) a[x >> 1].y = sA[buf][k * LDA + row];
      else a[x >> 1].x = sA[buf][k * LDA + row];
    } else if ((x & 1) == 0) {
      a[x >> 1] = *reinterpret_cast<const pd2*>(
          &sA[buf][row * PP_BK + 2 * ((2 * x + kq) ^ (row & 7))]);
    }
  };
  auto fetch_b = [&](int buf, int x, int j) {
    b[x & 1][j] = sB[buf][(8 * (x >> 1) + 2 * kq + (x & 1)) * LDB + 16 * j + m16];
  };
  Regs r0, r1;
  if (nst > 0) {
#pragma unroll
    for (int i = 0; i < NP; ++i) load(0, r0, i);
    if (nst > 1) {
#pragma unroll
      for (int i = 0; i < NP; ++i) load(1, r1, i);
    }
    zero_past_end(0, r0);
#pragma unroll
    for (int i = 0; i < NP; ++i) store(0, r0, i);
    if (nst > 2) {
#pragma unroll
      for (int i = 0; i < NP; ++i) load(2, r0, i);
    }
    __syncthreads();
    fetch_a(0, 0);
#pragma unroll
    for (int j = 0; j < WN; ++j) fetch_b(0, 0, j);
  }
  // k-tile st: its buffer is complete, its first operands are in registers,
  // k-tile st + 1 is in ``next`` and st + 2 on its way.  Each product's operands
  // are read while the one before runs; the barrier stands ahead of the last
  // product, which hides the waves' skew and the first reads of the next buffer.
  auto tile = [&](int st, Regs& next) {
    const int buf = st & 1;
    if (st + 1 < nst) {
      zero_past_end(st + 1, next);
#pragma unroll
      for (int i = 0; i < NP; ++i) store(st + 1, next, i);
    }
    if (st + 3 < nst) {
#pragma unroll
      for (int i = 0; i < NP; ++i) load(st + 3, next, i);
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      if (x == 3) __syncthreads();
      if (x < 3 || st + 1 < nst) {
        const int to = x < 3 ? buf : buf ^ 1;
        fetch_a(to, (x + 1) & 3);
#pragma unroll
        for (int j = 0; j < WN; ++j) fetch_b(to, (x + 1) & 3, j);
      }
      __builtin_amdgcn_sched_barrier(0);
      const double v = x & 1 ? a[x >> 1].y : a[x >> 1].x;
#pragma unroll
      for (int j = 0; j < WN; ++j)
        acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(v, b[x & 1][j], acc[j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  for (int st = 0; st < nst; st += 2) {
    tile(st, r1);
    if (st + 1 < nst) tile(st + 1, r0);
  }
#pragma unroll
  for (int j = 0; j < WN; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + 16 * wave + kq + 4 * r, n = n0 + 16 * j + m16;
      if (m >= g.M || n >= g.N) continue;
      const double v = acc[j][r];
      if (ksplit == 1) {
        const int64_t off = imap(g.cm, m) + imap(g.cn, n);
        C[off] = (g.beta != 0.0) ? g.alpha * v + g.beta * C[off] : g.alpha * v;
      } else {
        work[((int64_t)kpart * g.M + m) * g.N + n] = v;
      }
    }
}

// Small products (M, N and K each a few hundred at most): 64 x 64 tiles leave
// most CUs empty and every tile a serial chain over K (315 x 37 x 315: 5
// workgroups, 22.6 us; 66 x 66 x 1024 in 8 k parts: 12.8 us and a 4.4 us sum of
// the parts).  Here a workgroup owns one 16 x 16 tile and its waves (one for
// 64 k at most) each a run of k, read straight into registers in the matrix
// instruction's layout, four k steps a lane at a time; the waves' partial tiles are
// added in LDS in a fixed order.  Bound by two round trips to L2: 315 x 37 x
// 315 5.4 us, 66 x 66 x 1024 7.2 us.
// AK / BC: A's and B's k index has unit stride, so a lane's four steps are two
// 16-byte loads (their k order is free, the same for A and B).  GEN: any
// operand maps; the k parts of the addresses are evaluated once into LDS.
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));
constexpr int SP_U = 4;          // k blocks of 16 in flight per wave
constexpr int SP_MAXK = 3072;
template <bool AK, bool BC, bool GEN>
__global__ __launch_bounds__(1024) void gemm_f64_small_kernel(GemmDesc g, GemmBatch bt) {
  __shared__ double pool[GEN ? 2 * SP_MAXK : 16 * 256];
  if (g.run_if && *g.run_if == 0) return;
  const int tid = threadIdx.x, lane = tid & 63, nw = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = blockIdx.y * 16, n0 = blockIdx.x * 16;
  const int64_t sak = g.ak.s0, sbk = g.bk.s0;
  const int mr = min(m0 + (lane & 15), g.M - 1), nr = min(n0 + (lane & 15), g.N - 1);
  const double* __restrict__ pa = bt.A[blockIdx.z] + (GEN ? imap(g.am, mr) : mr * g.am.s0);
  const double* __restrict__ pb = bt.B[blockIdx.z] + (GEN ? imap(g.bn, nr) : nr * g.bn.s0);
  int64_t* koff = reinterpret_cast<int64_t*>(pool);
  if (GEN) {
    for (int e = tid; e < 2 * g.K; e += blockDim.x)
      koff[e] = e < g.K ? imap(g.ak, e) : imap(g.bk, e - g.K);
    __syncthreads();
  }
  auto a_at = [&](int k) { return pa[GEN ? koff[k] : k * sak]; };
  auto b_at = [&](int k) { return pb[GEN ? koff[g.K + k] : k * sbk]; };
  const int nb = (g.K + 15) / 16, kl = 4 * (lane >> 4);
  const int b0 = nb * wave / nw, b1 = nb * (wave + 1) / nw;
  d4 acc = {0.0, 0.0, 0.0, 0.0};
  for (int b = b0; b < b1; b += SP_U) {
    double a[SP_U][4], w[SP_U][4];
#pragma unroll
    for (int u = 0; u < SP_U; ++u) {
      if (b + u >= b1) continue;
      const int k = 16 * (b + u) + kl;
      if (16 * (b + u) + 16 <= g.K) {
        if (AK) {
          const d2u x = *(const d2u*)(pa + k), y = *(const d2u*)(pa + k + 2);
          a[u][0] = x[0]; a[u][1] = x[1]; a[u][2] = y[0]; a[u][3] = y[1];
        } else {
#pragma unroll
          for (int s = 0; s < 4; ++s) a[u][s] = a_at(k + s);
        }
        if (BC) {
          const d2u x = *(const d2u*)(pb + k), y = *(const d2u*)(pb + k + 2);
          w[u][0] = x[0]; w[u][1] = x[1]; w[u][2] = y[0]; w[u][3] = y[1];
        } else {
#pragma unroll
          for (int s = 0; s < 4; ++s) w[u][s] = b_at(k + s);
        }
      } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int kc = min(k + s, g.K - 1);
          a[u][s] = k + s < g.K ? a_at(kc) : 0.0;
          w[u][s] = k + s < g.K ? b_at(kc) : 0.0;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < SP_U; ++u) {
      if (b + u >= b1) continue;
#pragma unroll
      for (int s = 0; s < 4; ++s)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u][s], w[u][s], acc, 0, 0, 0);
    }
  }
  if (GEN) __syncthreads();  // the offsets have been read
#pragma unroll
  for (int r = 0; r < 4; ++r) pool[wave * 256 + r * 64 + lane] = acc[r];
  __syncthreads();
  for (int e = tid; e < 256; e += blockDim.x) {
    const int m = m0 + ((e & 63) >> 4) + 4 * (e >> 6), n = n0 + (e & 15);
    double v = pool[e];
    for (int w = 1; w < nw; ++w) v += pool[w * 256 + e];
    if (m >= g.M || n >= g.N) continue;
    double* C = bt.C[blockIdx.z];
    const int64_t off = imap(g.cm, m) + imap(g.cn, n);
    C[off] = (g.beta != 0.0) ? g.alpha * v + g.beta * C[off] : g.alpha * v;
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Shapes the pipelined kernel takes over: plainly strided as above (rows of even
// length: no 16-byte piece reaches past one) and large (gemm_f64_large).
bool pipe_shape(const GemmDesc& g, int count) {
  if (!g.pipe || count != 1) return false;
  if (g.am.n0 > 0 || g.ak.n0 > 0 || g.bk.n0 > 0 || g.bn.n0 > 0) return false;
  const bool am = g.am.s0 == 1 && g.ak.s0 != 1;
  if (!am && g.ak.s0 != 1) return false;
  const int64_t lda = am ? g.ak.s0 : g.am.s0, alen = am ? g.M : g.K;
  if (g.bn.s0 != 1 || ((lda | alen | g.bk.s0 | g.N) & 1)) return false;
  return gemm_f64_large(g.M, g.N, g.K);
}
int pipe_wn(const GemmDesc& g) {
  const int nt = (g.N + 16 * PP_MAXWN - 1) / (16 * PP_MAXWN);
  return ((g.N + nt - 1) / nt + 15) / 16;
}
// k parts: the fewest estimated microseconds of rounds of workgroups (two a CU,
// 512 WN clocks a k-tile for the pair) and of the partial sums' way through
// memory (about 4 TB/s, written and read).  Only the proportions matter, so the
// clock is the nominal 2.4 GHz, not the 2.2 that power leaves.
int pipe_ksplit(const GemmDesc& g) {
  const int wn = pipe_wn(g), kt = (g.K + PP_BK - 1) / PP_BK;
  const int64_t tiles = (int64_t)((g.M + PP_BM - 1) / PP_BM) * ((g.N + 16 * wn - 1) / (16 * wn));
  const double stage = 512.0 * wn / 2400.0, fixed = 5.0;
  int best = 1;
  double t_best = 0.0;
  for (int ks = 1; ks <= 64 && (ks == 1 || kt / ks >= 6); ++ks) {
    const int per = (kt + ks - 1) / ks;
    if (ks > 1 && (ks - 1) * per >= kt) continue;  // an empty part
    const double rounds = (double)((tiles * ks + 2048 / PP_NW - 1) / (2048 / PP_NW));
    double t = rounds * (per * stage + fixed);
    if (ks > 1) t += 4.0 + 2.0 * ks * g.M * (double)g.N * 8.0 / 4e6;
    if (ks == 1 || t < t_best) {
      best = ks;
      t_best = t;
    }
  }
  return best;
}

// Shapes the small kernel takes: within its range of K (102 x 102 x 2500: 15 us
// against 22, 16 x 16 x 4096: 24 against 16), not many tiles of next to no k
// (1000 x 1000 x 20: 12.6 us against 11.9), and up to 1.4e8 multiply-adds with the
// padding of its tiles, where reading the operands once a tile begins to cost
// more than the pipelined kernel's second launch (1024 x 66 x 1024: 15 - 17 us
// against 17.6 in two launches, 500^3: 16 against 24, 1600 x 72 x 1600: even, 8000 x
// 24 x 600: 26 against 19); one that the pipelined kernel takes in one launch
// stays there (1024 x 1024 x 64: 15.6 us against 16.2).
bool small_size(int64_t M, int64_t N, int64_t K, int count) {
  if (K <= 0 || K > SP_MAXK) return false;
  const int64_t tiles = (M + 15) / 16 * ((N + 15) / 16) * count;
  return 256.0 * tiles * K < 1.4e8 && tiles <= (K >= 32 ? 4096 : 1024);
}
bool small_shape(const GemmDesc& g, int count) {
  return g.pipe && small_size(g.M, g.N, g.K, count) &&
         (!pipe_shape(g, count) || pipe_ksplit(g) > 1);
}
void launch_small(const GemmDesc& g, const GemmBatch& b, hipStream_t s) {
  const dim3 grid((g.N + 15) / 16, (g.M + 15) / 16, b.count);
  const dim3 block(64 * std::min(16, std::max(1, (g.K + 63) / 64)));
  const bool lin = g.am.n0 <= 0 && g.ak.n0 <= 0 && g.bk.n0 <= 0 && g.bn.n0 <= 0;
  const bool ak = g.ak.s0 == 1, bc = g.bk.s0 == 1;
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, s, g, b); };
  if (!lin) launch(gemm_f64_small_kernel<false, false, true>);
  else if (ak && bc) launch(gemm_f64_small_kernel<true, true, false>);
  else if (ak) launch(gemm_f64_small_kernel<true, false, false>);
  else if (bc) launch(gemm_f64_small_kernel<false, true, false>);
  else launch(gemm_f64_small_kernel<false, false, false>);
}

template <int WN>
void launch_pipe_wn(const GemmDesc& g, const GemmBatch& b, int ks, double* work, hipStream_t s) {
  const dim3 grid((g.N + 16 * WN - 1) / (16 * WN), (g.M + PP_BM - 1) / PP_BM, ks);
  ACETN_REQUIRE(grid.y <= 65535 && grid.z <= 65535, "gemm_f64: grid too large");
  if (g.am.s0 == 1 && g.ak.s0 != 1)
    hipLaunchKernelGGL((gemm_f64_pipe_kernel<WN, true>), grid, dim3(PP_NT), 0, s, g, b.A[0], b.B[0],
                       b.C[0], ks, work);
  else
    hipLaunchKernelGGL((gemm_f64_pipe_kernel<WN, false>), grid, dim3(PP_NT), 0, s, g, b.A[0], b.B[0],
                       b.C[0], ks, work);
}
void launch_pipe(const GemmDesc& g, const GemmBatch& b, int ks, double* work, hipStream_t s) {
  switch (pipe_wn(g)) {
    case 2: launch_pipe_wn<2>(g, b, ks, work, s); break;
    case 3: launch_pipe_wn<3>(g, b, ks, work, s); break;
    case 4: launch_pipe_wn<4>(g, b, ks, work, s); break;
    case 5: launch_pipe_wn<5>(g, b, ks, work, s); break;
    case 6: launch_pipe_wn<6>(g, b, ks, work, s); break;
    case 7: launch_pipe_wn<7>(g, b, ks, work, s); break;
    case 8: launch_pipe_wn<8>(g, b, ks, work, s); break;
    case 9: launch_pipe_wn<9>(g, b, ks, work, s); break;
    default: launch_pipe_wn<10>(g, b, ks, work, s); break;
  }
}

// Small-output, long-K products (M, N <= 8, e.g. the d^2 x d^2 reduced
// density matrix summed over the whole environment): a 16 x 16 matrix-core
// tile would be almost all padding, so each lane walks its own k indices and
// accumulates all M x N dot products in registers; each workgroup reduces
// its lanes (shuffles, then LDS across waves) into one partial, and a second
// kernel sums the partials in a fixed order (bitwise reproducible).
constexpr int kDotMax = 8, kDotNT = 256, kDotWGs = 512, kDotMinK = 4096;

bool dot_small_fits(const GemmDesc& g) {
  return g.M <= kDotMax && g.N <= kDotMax && g.K >= kDotMinK;
}
int dot_small_wgs(const GemmDesc& g) {
  return (int)std::min<int64_t>(kDotWGs, ((int64_t)g.K + kDotNT - 1) / kDotNT);
}

__global__ __launch_bounds__(kDotNT) void dot_small_kernel(GemmDesc g, GemmBatch bt,
                                                           double* __restrict__ part) {
  constexpr int MN = kDotMax * kDotMax;
  __shared__ double red[kDotNT / 64][MN];
  if (g.run_if && *g.run_if == 0) return;
  const int prob = blockIdx.y;
  const double* __restrict__ A = bt.A[prob];
  const double* __restrict__ B = bt.B[prob];
  const int M = g.M, N = g.N;
  int64_t aoff[kDotMax], boff[kDotMax];
#pragma unroll
  for (int m = 0; m < kDotMax; ++m) aoff[m] = m < M ? imap(g.am, m) : 0;
#pragma unroll
  for (int n = 0; n < kDotMax; ++n) boff[n] = n < N ? imap(g.bn, n) : 0;
  double acc[kDotMax][kDotMax];
#pragma unroll
  for (int m = 0; m < kDotMax; ++m)
#pragma unroll
    for (int n = 0; n < kDotMax; ++n) acc[m][n] = 0.0;
  for (int k = blockIdx.x * kDotNT + threadIdx.x; k < g.K; k += gridDim.x * kDotNT) {
    const int64_t ka = imap(g.ak, k), kb = imap(g.bk, k);
    double a[kDotMax], b[kDotMax];
#pragma unroll
    for (int m = 0; m < kDotMax; ++m) a[m] = m < M ? A[aoff[m] + ka] : 0.0;
#pragma unroll
    for (int n = 0; n < kDotMax; ++n) b[n] = n < N ? B[kb + boff[n]] : 0.0;
#pragma unroll
    for (int m = 0; m < kDotMax; ++m)
#pragma unroll
      for (int n = 0; n < kDotMax; ++n) acc[m][n] = fma(a[m], b[n], acc[m][n]);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int m = 0; m < kDotMax; ++m)
#pragma unroll
    for (int n = 0; n < kDotMax; ++n) {
      double v = acc[m][n];
      for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o);
      if (lane == 0) red[wave][m * kDotMax + n] = v;
    }
  __syncthreads();
  if (threadIdx.x < MN) {
    double v = 0.0;
#pragma unroll
    for (int w = 0; w < kDotNT / 64; ++w) v += red[w][threadIdx.x];
    part[((int64_t)prob * gridDim.x + blockIdx.x) * MN + threadIdx.x] = v;
  }
}

// one workgroup per output element: strided partial sums, then a fixed
// binary tree in LDS (deterministic)
__global__ __launch_bounds__(kDotNT) void dot_small_reduce(GemmDesc g, GemmBatch bt,
                                                           const double* __restrict__ part,
                                                           int nwg) {
  constexpr int MN = kDotMax * kDotMax;
  __shared__ double red[kDotNT];
  if (g.run_if && *g.run_if == 0) return;
  const int prob = blockIdx.y, t = threadIdx.x;
  const int m = blockIdx.x / g.N, n = blockIdx.x % g.N;
  const double* p = part + (int64_t)prob * nwg * MN + m * kDotMax + n;
  double s = 0.0;
  for (int w = t; w < nwg; w += kDotNT) s += p[(int64_t)w * MN];
  red[t] = s;
  __syncthreads();
  for (int o = kDotNT / 2; o > 0; o >>= 1) {
    if (t < o) red[t] += red[t + o];
    __syncthreads();
  }
  if (t != 0) return;
  s = red[0];
  double* C = bt.C[prob];
  const int64_t off = imap(g.cm, m) + imap(g.cn, n);
  C[off] = (g.beta != 0.0) ? g.alpha * s + g.beta * C[off] : g.alpha * s;
}

struct Tile {
  int wm, wn;
  int var = 0;  // TuneChoice::var
};
int tile_bm(const Tile& t) { return 16 * t.wm * ((t.var & 1) ? 4 : 2); }
// per-shape tile: skinny range-finder products (N <= 160) use 64 x 160 / 32 x 160,
// large products 128 x 128, small ones 64 x 64
Tile choose_tile(const GemmDesc& g) {
  // skinny products: 64-row tiles only when K is long enough to split
  // (short-K products such as Y R^-1 need the tile count)
  if (g.N > 96 && g.N <= 160) return (g.M >= 2048 && g.K >= 1024) ? Tile{2, 5} : Tile{1, 5};
  if (g.M >= 1024 && g.N >= 1024) return Tile{4, 4};
  return Tile{2, 2};
}

int choose_ksplit_for(const GemmDesc& g, int count, const Tile& t) {
  const int BM = tile_bm(t), BN = 32 * t.wn;
  const int64_t tiles = (int64_t)((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN) * count;
  if (tiles >= 512 || g.K < 4 * BK * 8) return 1;
  int ks = (int)((1024 + tiles - 1) / tiles);
  ks = std::min(ks, g.K / (BK * 8));
  ks = std::min(ks, 64);
  return std::max(ks, 1);
}

int choose_ksplit(const GemmDesc& g, int count) {
  return choose_ksplit_for(g, count, choose_tile(g));
}

template <int WM, int WN>
void launch_gemm(const GemmDesc& g, const GemmBatch& b, int ks, double* work, hipStream_t s) {
  constexpr int BM = 32 * WM, BN = 32 * WN;
  dim3 grid((g.N + BN - 1) / BN, (g.M + BM - 1) / BM, b.count * ks);
  ACETN_REQUIRE(grid.y <= 65535 && grid.z <= 65535, "gemm_f64: grid too large");
  const bool lin = g.am.n0 <= 0 && g.ak.n0 <= 0 && g.bk.n0 <= 0 && g.bn.n0 <= 0;
  if (lin) hipLaunchKernelGGL((gemm_f64_kernel<WM, WN, true>), grid, dim3(NT), 0, s, g, b, ks, work);
  else hipLaunchKernelGGL((gemm_f64_kernel<WM, WN, false>), grid, dim3(NT), 0, s, g, b, ks, work);
}

// the wider WM x 5 variants (single-stride operand maps only)
template <int WM, int WGM, int BKT>
void launch_gemm_wide(const GemmDesc& g, const GemmBatch& b, int ks, double* work,
                      hipStream_t s) {
  constexpr int BM = 16 * WM * WGM, BN = 32 * 5;
  dim3 grid((g.N + BN - 1) / BN, (g.M + BM - 1) / BM, b.count * ks);
  ACETN_REQUIRE(grid.y <= 65535 && grid.z <= 65535, "gemm_f64: grid too large");
  hipLaunchKernelGGL((gemm_f64_kernel<WM, 5, true, WGM, BKT>), grid, dim3(128 * WGM), 0, s, g, b,
                     ks, work);
}
}  // namespace

// Large enough that 64-row tiles and a few k parts fill the chip: below 5e7
// products (324 x 38 x 324 has 4e6) a call is launches and latency either way.
bool gemm_f64_large(int64_t M, int64_t N, int64_t K) {
  return M >= 96 && N >= 17 && K >= 32 && (double)M * N * K >= 5e7;
}

int gemm_f64_size_limits(int64_t M, int64_t N, int64_t K, int count) {
  return (count == 1 && gemm_f64_large(M, N, K) ? kTuneNoPipe : 0) |
         (small_size(M, N, K, count) ? kTuneNoSmall : 0);
}

size_t gemm_f64_work_elems(const GemmDesc& g, int count) {
  if (dot_small_fits(g)) return (size_t)dot_small_wgs(g) * count * kDotMax * kDotMax;
  int ks = choose_ksplit(g, count);
  if (pipe_shape(g, count)) ks = std::max(ks, pipe_ksplit(g));
  return ks > 1 ? (size_t)ks * count * g.M * g.N : 0;
}

void gemm_f64(const GemmDesc& g, const GemmBatch& b, double* work, size_t work_elems,
              hipStream_t s) {
  ACETN_REQUIRE(b.count >= 1 && b.count <= kMaxBatch, "gemm_f64: bad batch count");
  if (g.M <= 0 || g.N <= 0) return;
  if (g.K <= 0) {
    // C = beta*C (or zero): handled by a K=1 product with zero contribution
    ACETN_REQUIRE(g.beta == 0.0, "gemm_f64: K == 0 with beta != 0 unsupported");
  }
  if (dot_small_fits(g) && work != nullptr &&
      work_elems >= (size_t)dot_small_wgs(g) * b.count * kDotMax * kDotMax) {
    const int nwg = dot_small_wgs(g);
    hipEvent_t e0 = kernel_timing_begin(s);
    hipLaunchKernelGGL(dot_small_kernel, dim3(nwg, b.count), dim3(kDotNT), 0, s, g, b, work);
    ACETN_HIP_CHECK(hipGetLastError());
    kernel_timing_end(e0, s, kKGemmF64, 2.0 * g.M * g.N * (double)g.K * b.count,
                      8.0 * ((double)g.M * g.K + (double)g.K * g.N + (double)g.M * g.N) * b.count);
    hipLaunchKernelGGL(dot_small_reduce, dim3(g.M * g.N, b.count), dim3(kDotNT), 0, s, g, b, work,
                       nwg);
    ACETN_HIP_CHECK(hipGetLastError());
    return;
  }
  auto fits = [&](int k) {
    return k == 1 || (work != nullptr && work_elems >= (size_t)k * b.count * g.M * g.N);
  };
  const bool lin = g.am.n0 <= 0 && g.ak.n0 <= 0 && g.bk.n0 <= 0 && g.bn.n0 <= 0;
  auto launch_choice = [&](const TuneChoice& c) {
    hipEvent_t e0 = kernel_timing_begin(s);
    if (c.wn == 1 && c.wm == 1) launch_small(g, b, s);
    else if (c.wn == 1) launch_pipe(g, b, c.ks, work, s);
    else if (c.wm == 2 && c.wn == 5 && lin && c.var == 1) launch_gemm_wide<2, 4, 16>(g, b, c.ks, work, s);
    else if (c.wm == 2 && c.wn == 5 && lin && c.var == 2) launch_gemm_wide<2, 2, 32>(g, b, c.ks, work, s);
    else if (c.wm == 2 && c.wn == 5 && lin && c.var == 3) launch_gemm_wide<2, 4, 32>(g, b, c.ks, work, s);
    else if (c.wm == 1 && c.wn == 5 && lin && c.var == 3) launch_gemm_wide<1, 4, 32>(g, b, c.ks, work, s);
    else if (c.wm == 2 && c.wn == 5) launch_gemm<2, 5>(g, b, c.ks, work, s);
    else if (c.wm == 1 && c.wn == 5) launch_gemm<1, 5>(g, b, c.ks, work, s);
    else if (c.wm == 4 && c.wn == 4) launch_gemm<4, 4>(g, b, c.ks, work, s);
    else launch_gemm<2, 2>(g, b, c.ks, work, s);
    ACETN_HIP_CHECK(hipGetLastError());
    kernel_timing_end(e0, s, kKGemmF64, 2.0 * g.M * g.N * (double)g.K * b.count,
                      8.0 * ((double)g.M * g.K + (double)g.K * g.N + (double)g.M * g.N) * b.count);
    if (c.ks > 1) {
      const int64_t mn = (int64_t)g.M * g.N;
      int blocks = (int)std::min<int64_t>((mn + 255) / 256, 2048);
      hipLaunchKernelGGL(splitk_reduce_kernel, dim3(blocks, b.count), dim3(256), 0, s, g, b, c.ks,
                         work);
      ACETN_HIP_CHECK(hipGetLastError());
    }
  };
  // A table entry holds for the products with its candidates: the sizes say
  // which of the pipelined and the small kernel there may be, the key which of
  // them this product may not take (order of sums, operand layout, alignment).
  const bool small = small_shape(g, b.count);
  const bool pipe = pipe_shape(g, b.count) && aligned16(b.A[0]) && aligned16(b.B[0]);
  const int limits = gemm_f64_size_limits(g.M, g.N, g.K, b.count) &
                     ~((pipe ? kTuneNoPipe : 0) | (small ? kTuneNoSmall : 0));
  const TuneKey key{0, g.M, g.N, g.K, (lin ? 1 : 0) | (b.count << 1) | limits};
  TuneChoice ch;
  const bool listed = autotune_lookup(key, &ch) && fits(ch.ks) && (ch.var == 0 || lin) &&
                      (ch.wn != 1 || (ch.wm == 1 ? small : pipe));
  if (!listed && autotune_should_tune(key, g, s)) {
    // The pipelined kernel leads: a tile that beats it by a few percent alone on
    // the GPU gains nothing beside other streams (5184 x 5184 x 144 on 64 x 64
    // tiles 194 - 199 us against 205; the FP64 iteration at D=6, chi=144 then 15.98 it/s
    // against 16.00 - 16.07), one that is far ahead does (2500 x 2500 x 100: 46
    // us against 59).
    std::vector<TuneChoice> cands;
    if (pipe) {
      const int h = pipe_ksplit(g);
      if (fits(h)) cands.push_back(TuneChoice{4, 1, h});
      if (h > 1) cands.push_back(TuneChoice{4, 1, 1});
    }
    const float lead = cands.empty() ? 1.f : 0.9f;
    if (small) cands.push_back(TuneChoice{1, 1, 1});
    const Tile tiles[8] = {{1, 5},    {2, 5},    {2, 2},    {4, 4},
                           {2, 5, 1}, {2, 5, 2}, {2, 5, 3}, {1, 5, 3}};
    for (const Tile& t : tiles) {
      if (t.var != 0 && !lin) continue;
      const int h = choose_ksplit_for(g, b.count, t);
      const int opts[4] = {1, h, 2 * h, h / 2};
      for (int k : opts) {
        if (k < 1 || k > 64 || !fits(k) || (k > 1 && g.K / k < 2 * BK)) continue;
        bool dup = false;
        for (const TuneChoice& c : cands)
          dup |= c.wm == t.wm && c.wn == t.wn && c.var == t.var && c.ks == k;
        if (dup) continue;
        TuneChoice c{t.wm, t.wn, k};
        c.var = t.var;
        cands.push_back(c);
      }
    }
    autotune_run(key, cands, s, launch_choice, lead);
    return;
  }
  if (!listed) {
    const Tile t = choose_tile(g);
    const int ks = choose_ksplit(g, b.count);
    ch = TuneChoice{t.wm, t.wn, fits(ks) ? ks : 1};
    const int parts = pipe && !small ? pipe_ksplit(g) : 0;
    if (small) ch = TuneChoice{1, 1, 1};
    else if (parts > 0 && fits(parts)) ch = TuneChoice{4, 1, parts};
  }
  launch_choice(ch);
}

GemmDesc dense_desc(int M, int N, int K, bool ta, int64_t lda, bool tb, int64_t ldb,
                    int64_t ldc, double alpha, double beta) {
  GemmDesc g{};
  g.M = M; g.N = N; g.K = K;
  g.am = ta ? plain(1) : plain(lda);
  g.ak = ta ? plain(lda) : plain(1);
  g.bk = tb ? plain(1) : plain(ldb);
  g.bn = tb ? plain(ldb) : plain(1);
  g.cm = plain(ldc);
  g.cn = plain(1);
  g.alpha = alpha;
  g.beta = beta;
  return g;
}

}  // namespace acetn
