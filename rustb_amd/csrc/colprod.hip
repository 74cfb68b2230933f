// Products of one k-point's n x n matrices (n <= 128) kept on chip: a
// workgroup of NT = ceil(n / 16) waves per k-point, wave J owning columns
// 16 J .. 16 J + 15 of every product.
//
//   T_J = X Z_J           A operand: X through LDS in 16-wide k-chunks, rows in
//                         groups of RT tiles (bounds the accumulators); B
//                         operand: the wave's own 16 columns of Z, from memory
//   C_IJ = Z_I^H T_J      A operand: 16 columns of Z through LDS per row tile
//                         I; B operand: T_J from the registers it was
//                         accumulated in
//
// The FP64 MFMA's accumulator register r of lane l holds D[4r + l/16][l%16],
// and its B operand is B[l/16][l%16]: with the k index of step r taken as
// 4r + l/16, an accumulator is the B operand of the next product as it stands,
// so T never leaves the registers and U^H X U costs one read of X and Z (and
// one of Z's columns) instead of a batched product's three matrices twice.
// The result is consumed by its epilogue or stored once.
//
// Complex products are 3M (three real MFMAs; planes re, im, re + im in LDS).
// Bound: the FP64 matrix cores (72 TFLOP/s of v_mfma_f64_16x16x4 on this
// device).  U^H M U with the band sum, 15798 k-points at n = 128: 6.7 ms, 59
// TFLOP/s executed (two batched products and the sum 8.9 ms); 131072 at n = 32:
// 1.5 ms (5.4 ms).
#include "eigh.hpp"
#include "gpu_team.hpp"

namespace rtb {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

__device__ inline d4 mfma64(double a, double b, d4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }

// How the first product reads X, and what becomes of the second.
enum : int {
  kMul = 0,    // T = X Z
  kMulH = 1,   // T = X^H Z
  kLoad = 2,   // T = X (its columns)
};
enum : int {
  kStore = 0,  // out[i][j] = C_ij
  kAbs2 = 1,   // out[i][j] = |C_ij|^2 (real)
  kKubo = 2,   // the one-product band sum: Omega from Q_ij = |C_ij|^2 / ((E_i - E_j)^2 + eta^2)
  kExact = 3,  // with P_ij = conj(A_ji) from a kStore pass, C = B: Omega, metric, diagonal
  kImK = 4,    // out[j][i] = Im(A_ji B_ij) (real)
};

struct ColArgs {
  int n;
  const double2* X;  // [nk] at stride sX
  size_t sX;
  const double2* Z;  // [nk][n][n] columns (also the left operand)
  const double* sc;  // [nk][n] column scales of Z, or null
  const double* E;   // [nk][n]
  double eta2;
  const double2* P;  // [nk][n][n]
  double2* out;      // [nk][n][n] complex (kStore)
  double* rout;      // [nk][n][n] real (kAbs2, kImK)
  double* omega;     // [nk][n]
  double* metric;    // [nk][n], or null
  double* diag;      // [nk][n] Re C_jj, or null
};

constexpr int kCK = 16;   // k-chunk of the first product
constexpr int kCLd = 17;  // its LDS row stride (doubles): rows on distinct banks

// Row tiles accumulated at a time in the first product: at NT = 8 two groups
// of 4 (96 accumulator registers beside the 128 of T).
template <int NT>
struct ColShape {
  static constexpr int RT = NT <= 4 ? NT : (NT <= 6 ? 3 : 4);
  static constexpr int NH = (NT + RT - 1) / RT;
  static constexpr int threads = 64 * NT;
  static constexpr size_t p1 = 3 * static_cast<size_t>(16 * RT) * kCLd;  // doubles per buffer
  static constexpr size_t p2 = 3 * static_cast<size_t>(16 * NT) * 16;
  static constexpr size_t buf = 2 * (p1 > p2 ? p1 : p2);
  // after the buffers: E, scale [16 NT], row sums [NT][16 NT]
  static constexpr size_t doubles = buf + 2 * 16 * NT + static_cast<size_t>(NT) * 16 * NT;
};

// T_J = X Z_J (or X^H Z_J) of the wave's 16 columns: tr, ti[K][r] = T[16 K + 4 r +
// fk][col].  smem: two buffers of ColShape::p1 doubles; Z's columns in FP64 or
// FP32 (exact).
template <int NT, int OP, typename ZT>
__device__ __forceinline__ void first_product(double* smem, const double2* __restrict__ X, const ZT* __restrict__ Z,
                                              int n, int tid, int fr, int fk, int col, double (&tr)[NT][4],
                                              double (&ti)[NT][4]) {
  using Sh = ColShape<NT>;
  constexpr int RT = Sh::RT, NH = Sh::NH, TH = Sh::threads;
  constexpr int EL = (16 * RT * kCK + TH - 1) / TH;  // staged elements per thread
  constexpr int PL = 16 * RT * kCLd;                 // plane
  const int nc = (n + kCK - 1) / kCK;
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    const int r0 = 16 * RT * h;
    double2 px[EL];
    ZT pb[4];
    // outside the matrix: any entry of it (a row i >= n of the product is
    // not used, a column k >= n meets a zero row of Z)
    const auto load_x = [&](int k0) {
#pragma unroll
      for (int u = 0; u < EL; ++u) {
        const int q = tid + TH * u;
        if constexpr (OP == kMul) {  // lanes along k within a row
          const int i = min(r0 + q / kCK, n - 1), k = min(k0 + q % kCK, n - 1);
          px[u] = X[static_cast<unsigned>(i * n + k)];
        } else {  // X^H: lanes along the row of X
          const int k = min(k0 + q / (16 * RT), n - 1), i = min(r0 + q % (16 * RT), n - 1);
          px[u] = X[static_cast<unsigned>(k * n + i)];
        }
      }
    };
    const auto store_x = [&](double* b) {
#pragma unroll
      for (int u = 0; u < EL; ++u) {
        const int q = tid + TH * u;
        if (16 * RT * kCK % TH == 0 || q < 16 * RT * kCK) {
          const int i = OP == kMul ? q / kCK : q % (16 * RT), k = OP == kMul ? q % kCK : q / (16 * RT);
          const double re = px[u].x, im = OP == kMul ? px[u].y : -px[u].y;
          b[i * kCLd + k] = re;
          b[PL + i * kCLd + k] = im;
          b[2 * PL + i * kCLd + k] = re + im;
        }
      }
    };
    const auto load_b = [&](int k0) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int k = k0 + 4 * s + fk;
        pb[s] = Z[static_cast<unsigned>(min(k, n - 1) * n + min(col, n - 1))];
      }
    };
    d4 a1[RT], a2[RT], a3[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) a1[t] = a2[t] = a3[t] = d4{0.0, 0.0, 0.0, 0.0};
    load_x(0);
    load_b(0);
    if (h > 0) __syncthreads();  // the previous group's last chunk is consumed
    store_x(smem);
    if (nc > 1) load_x(kCK);
    __syncthreads();
    // chunk c from buffer c % 2; in its middle the next chunk, loaded a whole
    // chunk earlier, goes to the other buffer, so the barrier at the end finds
    // it written
#pragma unroll 1
    for (int c = 0; c < nc; ++c) {
      const double* b = smem + (c & 1) * Sh::p1;
      double br[4], bi[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const bool in = kCK * c + 4 * s + fk < n && col < n;  // (here, not at the load: a use waits for it)
        br[s] = in ? static_cast<double>(pb[s].x) : 0.0;
        bi[s] = in ? static_cast<double>(pb[s].y) : 0.0;
      }
      if (c + 1 < nc) load_b((c + 1) * kCK);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (s == 2 && c + 1 < nc) {
          store_x(smem + ((c + 1) & 1) * Sh::p1);
          if (c + 2 < nc) load_x((c + 2) * kCK);
        }
        const double bs = br[s] + bi[s];
        const double* f = b + fr * kCLd + 4 * s + fk;
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          if (RT * h + t < NT) {
            const double* g = f + 16 * t * kCLd;
            a1[t] = mfma64(g[0], br[s], a1[t]);
            a2[t] = mfma64(g[PL], bi[s], a2[t]);
            a3[t] = mfma64(g[2 * PL], bs, a3[t]);
          }
          if (NT >= 7 && t % 2 == 1) __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_sched_barrier(0);  // bounded look-ahead of the LDS reads (registers)
      }
      if (c + 1 < nc) __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < RT; ++t)
      if (RT * h + t < NT) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          tr[RT * h + t][r] = a1[t][r] - a2[t][r];
          ti[RT * h + t][r] = a3[t][r] - a1[t][r] - a2[t][r];
        }
      }
  }
}

template <int NT, int OP, int EP>
__global__ void __launch_bounds__(64 * NT) __attribute__((amdgpu_waves_per_eu(2))) col_product_kernel(ColArgs a) {
  using Sh = ColShape<NT>;
  constexpr int TH = Sh::threads, N = 16 * NT;
  extern __shared__ __align__(16) double smem[];
  double* sE = smem + Sh::buf;
  double* sS = sE + N;
  double* sRow = sS + N;  // [NT][N]
  const int n = a.n;
  const size_t mat = blockIdx.x;
  const size_t nn = static_cast<size_t>(n) * n;
  const double2* __restrict__ X = a.X + mat * a.sX;
  const double2* __restrict__ Z = a.Z + mat * nn;
  const double2* __restrict__ P = a.P + mat * nn;  // kExact, kImK
  const int tid = threadIdx.x, lane = tid & 63;
  const int J = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fk = lane >> 4;
  const int col = 16 * J + fr;
  for (int i = tid; i < N; i += TH) {
    sE[i] = a.E && i < n ? a.E[mat * n + i] : 0.0;
    sS[i] = a.sc && i < n ? a.sc[mat * n + i] : 1.0;
  }
  // ---- T_J ----
  double tr[NT][4], ti[NT][4];
  if constexpr (OP == kLoad) {
#pragma unroll
    for (int K = 0; K < NT; ++K)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = 16 * K + 4 * r + fk;
        const double2 x = k < n && col < n ? X[static_cast<unsigned>(k * n + col)] : make_double2(0.0, 0.0);
        tr[K][r] = x.x;
        ti[K][r] = x.y;
      }
  } else {
    first_product<NT, OP>(smem, X, Z, n, tid, fr, fk, col, tr, ti);
  }
  // ---- C_IJ = Z_I^H T_J, row tile by row tile ----
  constexpr int EL2 = 16 * N / TH;  // 4
  double2 pz[EL2];
  auto load2 = [&](int I) {
#pragma unroll
    for (int u = 0; u < EL2; ++u) {
      const int q = tid + TH * u;
      const int k = q / 16, c = min(16 * I + q % 16, n - 1);
      pz[u] = Z[static_cast<unsigned>(min(k, n - 1) * n + c)];
    }
  };
  const auto store2 = [&](double* b) {
#pragma unroll
    for (int u = 0; u < EL2; ++u) {
      const int q = tid + TH * u;
      const bool in = q / 16 < n;  // rows of T past n are not zero
      const double re = in ? pz[u].x : 0.0, im = in ? -pz[u].y : 0.0;  // Z^H
      b[q] = re;
      b[16 * N + q] = im;
      b[2 * 16 * N + q] = re + im;
    }
  };
  double colsum = 0.0, colsum2 = 0.0;  // Omega (column sum of Q), metric
  load2(0);
  __syncthreads();  // the first product's buffers are free; sE, sS are visible
  store2(smem);
  if (NT > 1) load2(1);
  __syncthreads();
  const double Ej = sE[col], sj = sS[col];
#pragma unroll 1
  for (int I = 0; I < NT; ++I) {
    const double* b = smem + (I & 1) * Sh::p2;
    double2 pp[4];
    if constexpr (EP == kExact || EP == kImK) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * I + 4 * r + fk;
        pp[r] = P[static_cast<unsigned>(min(i, n - 1) * n + min(col, n - 1))];
      }
    }
    d4 c1 = {0.0, 0.0, 0.0, 0.0}, c2 = c1, c3 = c1;
#pragma unroll
    for (int K = 0; K < NT; ++K) {
      if (K == NT / 2 && I + 1 < NT) {  // the next row tile, as in first_product
        store2(smem + ((I + 1) & 1) * Sh::p2);
        if (I + 2 < NT) load2(I + 2);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double* g = b + (16 * K + 4 * r + fk) * 16 + fr;
        c1 = mfma64(g[0], tr[K][r], c1);
        c2 = mfma64(g[16 * N], ti[K][r], c2);
        c3 = mfma64(g[2 * 16 * N], tr[K][r] + ti[K][r], c3);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    double rowq[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * I + 4 * r + fk;
      double re = c1[r] - c2[r], im = c3[r] - c1[r] - c2[r];
      rowq[r] = 0.0;
      const bool in = i < n && col < n;
      const size_t o = mat * nn + static_cast<size_t>(i) * n + col;
      if constexpr (EP != kAbs2) {
        if (a.sc) {
          const double f = sS[i] * sj;
          re *= f;
          im *= f;
        }
      }
      if constexpr (EP == kStore) {
        if (in) a.out[o] = make_double2(re, im);
      } else if constexpr (EP == kAbs2) {
        if (in) a.rout[o] = re * re + im * im;
      } else if constexpr (EP == kKubo) {
        if (in && i != col) {
          // 1 / (d^2 + eta^2): hardware reciprocal and two Newton steps
          const double d = sE[i] - Ej;
          const double den = fma(d, d, a.eta2);
          double rc = __builtin_amdgcn_rcp(den);
          rc = fma(rc, fma(-den, rc, 1.0), rc);
          rc = fma(rc, fma(-den, rc, 1.0), rc);
          const double q = (re * re + im * im) * rc;
          colsum += q;
          rowq[r] = q;
        }
      } else if constexpr (EP == kExact) {
        // A_ji B_ij with A_ji = conj(P_ij)
        if (in && i != col) {
          const double d = Ej - sE[i];
          const double den = d * d + a.eta2;
          colsum += -2.0 * (pp[r].x * im - pp[r].y * re) / den;
          if (a.metric) colsum2 += (pp[r].x * re + pp[r].y * im) / den;
        }
        if (a.diag && in && i == col) a.diag[mat * n + col] = re;
      } else {  // kImK
        if (in) a.rout[mat * nn + static_cast<size_t>(col) * n + i] = pp[r].x * im - pp[r].y * re;
      }
    }
    if constexpr (EP == kKubo) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double x = row_sum16(rowq[r]);  // the wave's 16 columns of row i
        if (fr == 0) sRow[J * N + 16 * I + 4 * r + fk] = x;
      }
    }
    if (I + 1 < NT) __syncthreads();
  }
  if constexpr (EP == kKubo || EP == kExact) {
    colsum += __shfl_xor(colsum, 16, 64);
    colsum += __shfl_xor(colsum, 32, 64);
    if constexpr (EP == kKubo) {
      __syncthreads();
      if (fk == 0 && col < n) {
        double row = 0.0;
#pragma unroll
        for (int w = 0; w < NT; ++w) row += sRow[w * N + col];
        a.omega[mat * n + col] = 0.5 * (colsum - row);
      }
    } else {
      if (fk == 0 && col < n) a.omega[mat * n + col] = colsum;
      if (a.metric) {  // uniform
        colsum2 += __shfl_xor(colsum2, 16, 64);
        colsum2 += __shfl_xor(colsum2, 32, 64);
        if (fk == 0 && col < n) a.metric[mat * n + col] = colsum2;
      }
    }
  }
}

// ---- the refinement of FP32 eigenpairs, one k-point per workgroup ----
// One Ogita-Aishima step (see refine_eigenpairs) without leaving the chip:
//   HZ_J = H Z_J                              FP64 MFMA
//   lt_j = Re z_j^H (HZ)_j / |z_j|^2, R_J = HZ_J - Z_J diag(lt)
//   F_J  = off-diagonal (Z^H R)_ij / (lt_j - lt_i)   FP64 MFMA
// which is (S_ij - lt_j G_ij) / (lt_j - lt_i) for S = Z^H H Z, G = Z^H Z: one
// product instead of two, with the cancellation done before it.  Inside
// clusters F_ij = -G_ij / 2, a dot product for those pairs; F_jj = (1 - G_jj) / 2.
//   D_J = Z F_J, HD_J = H D_J                 FP32 MFMA (F is of the size of
//                                             the FP32 vectors' error)
//   z' = z + d, r' = (H - lt) z' = R + HD - lt D,
//   E_j = lt_j + Re z'^H r' / |z'|^2, residual |r'| / |z'|.
// HZ, F and D are used from registers: their layouts are the next product's B operand
// (the FP32 accumulator's rows 4 fk + r are made the FP64 one's 4 r + fk by
// giving lane row m of the A operand matrix row 4 (m % 4) + m / 4).  R is
// parked in memory over the FP32 products, F passes through memory between
// the loops that make and use it (registers: one tile of F at a time keeps
// those loops rolled).  LDS: k-chunks of H, then Z in FP32 with a k-chunk of H
// beside it (160 KB at NT = 8).
// Bound: the matrix cores (FP64 2 x 3M, FP32 2 x 3M products per k-point), at
// NT = 8 with one workgroup per CU, whose phases nothing else covers: n = 128,
// 15798 k-points 13.5 ms (FP64 products, Gram epilogue and FP32 corrections as
// batched kernels 16.4 ms); n = 32, 131072 k-points 3.4 ms (12.3 ms).
typedef float f4 __attribute__((ext_vector_type(4)));
__device__ inline f4 mfma32(float a, float b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

template <int NT>
struct RefShape {
  static constexpr int N = 16 * NT, threads = 64 * NT;
  static constexpr int zld = N + 1;  // complex FP32 row stride of Z
  static constexpr size_t z = static_cast<size_t>(N) * zld;                    // doubles (8 bytes per element)
  static constexpr size_t p1 = 2 * ColShape<NT>::p1;
  static constexpr size_t h = 3 * static_cast<size_t>(N) * kCLd / 2;           // a chunk of H in FP32 planes
  static constexpr size_t buf = z + h > p1 ? z + h : p1;
  static constexpr size_t doubles = buf + 2 * N;                               // lt, gd
};

template <int NT>
__global__ void __launch_bounds__(64 * NT) __attribute__((amdgpu_waves_per_eu(2))) refine_cols_kernel(
    int n, const double2* __restrict__ Hg, const float2* __restrict__ Zg, double2* __restrict__ Wg,
    double2* __restrict__ Zpg, double* __restrict__ E, double* __restrict__ scale, double* __restrict__ resid,
    double gap_rel) {
  using Sh = RefShape<NT>;
  constexpr int N = Sh::N, TH = Sh::threads, ZL = Sh::zld;
  extern __shared__ __align__(16) double smem[];
  double* sLt = smem + Sh::buf;
  double* sGd = sLt + N;
  const size_t mat = blockIdx.x;
  const size_t nn = static_cast<size_t>(n) * n;
  const double2* __restrict__ H = Hg + mat * nn;
  const float2* __restrict__ Z = Zg + mat * nn;
  double2* __restrict__ W = Wg + mat * nn;
  const int tid = threadIdx.x, lane = tid & 63;
  const int J = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fk = lane >> 4;
  const int col = 16 * J + fr;
  const int pr = 4 * (fr & 3) + (fr >> 2);  // matrix row of lane row fr in the FP32 products
  for (int i = tid; i < N; i += TH) sGd[i] = i < n ? scale[mat * n + i] : 1.0;
  double tr[NT][4], ti[NT][4];
  first_product<NT, kMul>(smem, H, Z, n, tid, fr, fk, col, tr, ti);
  // offset of the wave's element (K, r), clamped into the matrix
  const int cc = min(col, n - 1);
  // (nv: n, made opaque per loop so that the offsets of one loop do not stay
  // in registers for the next)
  const auto at = [&](int K, int r, int nv) { return static_cast<unsigned>(min(16 * K + 4 * r + fk, nv - 1) * nv + cc); };
  const auto opaque = [](int x) {
    asm volatile("" : "+s"(x));
    return x;
  };
  const auto inside = [&](int K, int r) { return 16 * K + 4 * r + fk < n && col < n; };
  double s = 0.0;
  int nv = opaque(n);
#pragma unroll
  for (int K = 0; K < NT; ++K)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float2 z = Z[at(K, r, nv)];
      const double x = fma(static_cast<double>(z.x), tr[K][r], static_cast<double>(z.y) * ti[K][r]);
      s += inside(K, r) ? x : 0.0;
    }
  s += __shfl_xor(s, 16, 64);
  s += __shfl_xor(s, 32, 64);
  __syncthreads();  // sGd is visible; the H chunks are consumed
  const double lt = col < n ? s / sGd[col] : 0.0;
  if (fk == 0) sLt[col] = lt;
  // R = HZ - lt Z, parked
  nv = opaque(n);
#pragma unroll
  for (int K = 0; K < NT; ++K) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float2 z = Z[at(K, r, nv)];
      tr[K][r] = fma(-lt, static_cast<double>(z.x), tr[K][r]);
      ti[K][r] = fma(-lt, static_cast<double>(z.y), ti[K][r]);
      if (inside(K, r)) W[at(K, r, nv)] = make_double2(tr[K][r], ti[K][r]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // Z into LDS (zero outside the matrix)
  float2* sZ = reinterpret_cast<float2*>(smem);
#pragma unroll 8
  for (int q = tid; q < N * N; q += TH) {
    const int i = q / N, c = q % N;
    const float2 z = Z[static_cast<unsigned>(min(i, n - 1) * n + min(c, n - 1))];
    sZ[i * ZL + c] = i < n && c < n ? z : make_float2(0.f, 0.f);
  }
  __syncthreads();
  double mx = 0.0;
  for (int i = lane; i < n; i += 64) mx = fmax(mx, fabs(sLt[i]));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
  const double thr = gap_rel * fmax(mx, 1.0);
  const double gdj = sGd[col];
  // F_J, row tile by row tile; it waits in the slots of Z' (FP32)
  double2* __restrict__ Zp = Zpg + mat * nn;
#pragma unroll 1
  for (int I = 0; I < NT; ++I) {
    d4 c1 = {0.0, 0.0, 0.0, 0.0}, c2 = c1, c3 = c1;
#pragma unroll
    for (int K = 0; K < NT; ++K) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float2 z = sZ[(16 * K + 4 * r + fk) * ZL + 16 * I + fr];  // Z^H: conjugated
        const double ar = z.x, ai = -z.y;
        c1 = mfma64(ar, tr[K][r], c1);
        c2 = mfma64(ai, ti[K][r], c2);
        c3 = mfma64(ar + ai, tr[K][r] + ti[K][r], c3);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll 1
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * I + 4 * r + fk;
      const double a1 = r == 0 ? c1[0] : (r == 1 ? c1[1] : (r == 2 ? c1[2] : c1[3]));
      const double a2 = r == 0 ? c2[0] : (r == 1 ? c2[1] : (r == 2 ? c2[2] : c2[3]));
      const double a3 = r == 0 ? c3[0] : (r == 1 ? c3[1] : (r == 2 ? c3[2] : c3[3]));
      const double re = a1 - a2, im = a3 - a1 - a2;
      const double dl = lt - sLt[i];
      const bool in = i < n && col < n;
      const bool near = in && i != col && !(fabs(dl) > thr);
      const double inv = 1.0 / dl;
      double f = re * inv, g = im * inv;
      if (__any(near)) {  // a cluster: -G_ij / 2 (exact FP32 products, FP64 sums)
        double gr = 0.0, gi = 0.0;
        for (int k = 0; k < n; ++k) {
          const float2 a = sZ[k * ZL + i], b = sZ[k * ZL + col];
          const double ax = a.x, ay = a.y, bx = b.x, by = b.y;
          gr += ax * bx + ay * by;
          gi += ax * by - ay * bx;
        }
        if (near) {
          f = -0.5 * gr;
          g = -0.5 * gi;
        }
      }
      if (i == col) {
        f = 0.5 * (1.0 - gdj);
        g = 0.0;
      }
      if (in)
        *reinterpret_cast<float2*>(&Zp[static_cast<unsigned>(i * n + col)]) =
            make_float2(static_cast<float>(f), static_cast<float>(g));
    }
  }
  float Fr[NT][4], Fi[NT][4];
  nv = opaque(n);
#pragma unroll
  for (int K = 0; K < NT; ++K)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float2 f = *reinterpret_cast<const float2*>(&Zp[at(K, r, nv)]);
      Fr[K][r] = inside(K, r) ? f.x : 0.f;
      Fi[K][r] = inside(K, r) ? f.y : 0.f;
    }
  // row tile I of D_J = Z F_J, which is the B operand of H's k-chunk I for
  // HD_J = H D_J (the chunk in FP32 planes, all row tiles); z' = z + d
  constexpr int EL = N * kCK / TH;  // 4
  float* sH = reinterpret_cast<float*>(smem + Sh::z);
  constexpr int PL = N * kCLd;      // plane
  double2 ph[EL];
  const auto load = [&](int k0) {
#pragma unroll
    for (int u = 0; u < EL; ++u) {
      const int q = tid + TH * u;
      ph[u] = H[static_cast<unsigned>(min(q / kCK, n - 1) * n + min(k0 + q % kCK, n - 1))];
    }
  };
  f4 h1[NT], h2[NT], h3[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) h1[t] = h2[t] = h3[t] = f4{0.f, 0.f, 0.f, 0.f};
  double den = 0.0;
  load(0);
#pragma unroll 1
  for (int I = 0; I < NT; ++I) {
    if (I > 0) __syncthreads();  // the previous chunk of H is consumed
#pragma unroll
    for (int u = 0; u < EL; ++u) {
      const int q = tid + TH * u;
      const int i = q / kCK, k = q % kCK;
      const float re = static_cast<float>(ph[u].x), im = static_cast<float>(ph[u].y);
      sH[i * kCLd + k] = re;
      sH[PL + i * kCLd + k] = im;
      sH[2 * PL + i * kCLd + k] = re + im;
    }
    if (I + 1 < NT) load(16 * (I + 1));
    float2 zo[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) zo[r] = Z[static_cast<unsigned>(min(16 * I + 4 * r + fk, n - 1) * n + cc)];
    f4 c1 = {0.f, 0.f, 0.f, 0.f}, c2 = c1, c3 = c1;
    const float2* zr = sZ + (16 * I + pr) * ZL + fk;
#pragma unroll
    for (int K = 0; K < NT; ++K) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float2 z = zr[16 * K + 4 * r];
        c1 = mfma32(z.x, Fr[K][r], c1);
        c2 = mfma32(z.y, Fi[K][r], c2);
        c3 = mfma32(z.x + z.y, Fr[K][r] + Fi[K][r], c3);
      }
      if (K % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();  // the chunk of H is written
    float dr[4], di[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      dr[r] = c1[r] - c2[r];
      di[r] = c3[r] - c1[r] - c2[r];
      const int k = 16 * I + 4 * r + fk;
      const unsigned o = static_cast<unsigned>(min(k, n - 1) * n + cc);
      const float2 z = zo[r];
      if (k < n && col < n) {
        const double zr1 = static_cast<double>(z.x) + dr[r], zi1 = static_cast<double>(z.y) + di[r];
        Zp[o] = make_double2(zr1, zi1);
        den += zr1 * zr1 + zi1 * zi1;
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float bs = dr[r] + di[r];
      const float* f = sH + pr * kCLd + 4 * r + fk;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        h1[t] = mfma32(f[16 * t * kCLd], dr[r], h1[t]);
        h2[t] = mfma32(f[PL + 16 * t * kCLd], di[r], h2[t]);
        h3[t] = mfma32(f[2 * PL + 16 * t * kCLd], bs, h3[t]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // r' = R + HD - lt D (D = z' - z) and the column sums
  double num = 0.0, res = 0.0;
  nv = opaque(n);
#pragma unroll
  for (int K = 0; K < NT; ++K) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const unsigned o = at(K, r, nv);
      const float2 z = Z[o];
      const double2 w = W[o], zp = Zp[o];
      const double p1 = h1[K][r], p2 = h2[K][r], p3 = h3[K][r];
      const double rr = fma(-lt, zp.x - z.x, w.x + (p1 - p2)), ri = fma(-lt, zp.y - z.y, w.y + (p3 - p1 - p2));
      if (inside(K, r)) {
        num += zp.x * rr + zp.y * ri;
        res += rr * rr + ri * ri;
      }
    }
    if (K % 2 == 1) __builtin_amdgcn_sched_barrier(0);
  }
  den += __shfl_xor(den, 16, 64);
  den += __shfl_xor(den, 32, 64);
  num += __shfl_xor(num, 16, 64);
  num += __shfl_xor(num, 32, 64);
  res += __shfl_xor(res, 16, 64);
  res += __shfl_xor(res, 32, 64);
  if (fk == 0 && col < n) {
    E[mat * n + col] = lt + num / den;
    scale[mat * n + col] = 1.0 / sqrt(den);
    resid[mat * n + col] = sqrt(res / den);
  }
}

template <int NT>
int launch_refine(hipStream_t st, int n, size_t nk, const double* H, const float* Z, double* W1, double* W2,
                  double* E, double* scale, double* resid, double gap_rel) {
  hipLaunchKernelGGL((refine_cols_kernel<NT>), dim3(static_cast<unsigned>(nk)), dim3(64 * NT),
                     RefShape<NT>::doubles * sizeof(double), st, n, reinterpret_cast<const double2*>(H),
                     reinterpret_cast<const float2*>(Z), reinterpret_cast<double2*>(W1),
                     reinterpret_cast<double2*>(W2), E, scale, resid, gap_rel);
  RTB_HIP(hipGetLastError());
  return RTB_OK;
}
template <int NT>
int refine_limit() {
  RTB_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&refine_cols_kernel<NT>),
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              static_cast<int>(RefShape<NT>::doubles * sizeof(double))));
  return RTB_OK;
}

template <int NT, int OP, int EP>
int launch_nt(hipStream_t st, size_t nk, const ColArgs& a) {
  constexpr size_t smem = ColShape<NT>::doubles * sizeof(double);
  hipLaunchKernelGGL((col_product_kernel<NT, OP, EP>), dim3(static_cast<unsigned>(nk)), dim3(64 * NT), smem, st, a);
  RTB_HIP(hipGetLastError());
  return RTB_OK;
}

template <int OP, int EP>
int launch_col(hipStream_t st, size_t nk, const ColArgs& a) {
  if (nk == 0) return RTB_OK;
  if (a.n < 1 || a.n > kMaxEighN) return fail(RTB_ERR_UNSUPPORTED, "column products are for 1 <= nsta <= 128");
  if (nk > 0x7fffffffu) return fail(RTB_ERR_UNSUPPORTED, "too many k-points in one launch");
  switch ((a.n + 15) / 16) {
    case 1: return launch_nt<1, OP, EP>(st, nk, a);
    case 2: return launch_nt<2, OP, EP>(st, nk, a);
    case 3: return launch_nt<3, OP, EP>(st, nk, a);
    case 4: return launch_nt<4, OP, EP>(st, nk, a);
    case 5: return launch_nt<5, OP, EP>(st, nk, a);
    case 6: return launch_nt<6, OP, EP>(st, nk, a);
    case 7: return launch_nt<7, OP, EP>(st, nk, a);
    default: return launch_nt<8, OP, EP>(st, nk, a);
  }
}

template <int NT, int OP, int EP>
int col_limit() {
  RTB_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&col_product_kernel<NT, OP, EP>),
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              static_cast<int>(ColShape<NT>::doubles * sizeof(double))));
  return RTB_OK;
}
template <int OP, int EP>
int col_limits() {  // NT >= 5 takes more than 64 KB
  RTB_TRY((col_limit<5, OP, EP>()));
  RTB_TRY((col_limit<6, OP, EP>()));
  RTB_TRY((col_limit<7, OP, EP>()));
  RTB_TRY((col_limit<8, OP, EP>()));
  return RTB_OK;
}

ColArgs col_args(int n, const double* X, size_t sX, const double* Z, const double* sc) {
  ColArgs a{};
  a.n = n;
  a.X = reinterpret_cast<const double2*>(X);
  a.sX = sX;
  a.Z = reinterpret_cast<const double2*>(Z);
  a.sc = sc;
  return a;
}

}  // namespace

int col_kubo(hipStream_t st, int n, size_t nk, const double* M, const double* Z, const double* sc, const double* E,
             double eta, double* omega) {
  ColArgs a = col_args(n, M, static_cast<size_t>(n) * n, Z, sc);
  a.E = E;
  a.eta2 = eta * eta;
  a.omega = omega;
  return launch_col<kMul, kKubo>(st, nk, a);
}

int col_project_adjoint(hipStream_t st, int n, size_t nk, const double* X, size_t sX, const double* Z,
                        const double* sc, double* P) {
  ColArgs a = col_args(n, X, sX, Z, sc);
  a.out = reinterpret_cast<double2*>(P);
  return launch_col<kMulH, kStore>(st, nk, a);
}

int col_kubo_exact(hipStream_t st, int n, size_t nk, const double* X, size_t sX, const double* Z, const double* sc,
                   const double* P, const double* E, double eta, double* omega, double* metric, double* diag) {
  ColArgs a = col_args(n, X, sX, Z, sc);
  a.P = reinterpret_cast<const double2*>(P);
  a.E = E;
  a.eta2 = eta * eta;
  a.omega = omega;
  a.metric = metric;
  a.diag = diag;
  return launch_col<kMul, kExact>(st, nk, a);
}

int col_im_k(hipStream_t st, int n, size_t nk, const double* X, size_t sX, const double* Z, const double* P,
             double* Ki) {
  ColArgs a = col_args(n, X, sX, Z, nullptr);
  a.P = reinterpret_cast<const double2*>(P);
  a.rout = Ki;
  return launch_col<kMul, kImK>(st, nk, a);
}

int col_overlap2(hipStream_t st, int n, size_t nk, const double* Ui, const double* Uj, double* out) {
  ColArgs a = col_args(n, Uj, static_cast<size_t>(n) * n, Ui, nullptr);
  a.rout = out;
  return launch_col<kLoad, kAbs2>(st, nk, a);
}

int col_refine(hipStream_t st, int n, size_t nk, const double* H, const float* Z, double* W1, double* W2, double* E,
               double* scale, double* resid, double gap_rel) {
  if (nk == 0) return RTB_OK;
  if (n < 1 || n > kMaxEighN) return fail(RTB_ERR_UNSUPPORTED, "column products are for 1 <= nsta <= 128");
  if (nk > 0x7fffffffu) return fail(RTB_ERR_UNSUPPORTED, "too many k-points in one launch");
  switch ((n + 15) / 16) {
    case 1: return launch_refine<1>(st, n, nk, H, Z, W1, W2, E, scale, resid, gap_rel);
    case 2: return launch_refine<2>(st, n, nk, H, Z, W1, W2, E, scale, resid, gap_rel);
    case 3: return launch_refine<3>(st, n, nk, H, Z, W1, W2, E, scale, resid, gap_rel);
    case 4: return launch_refine<4>(st, n, nk, H, Z, W1, W2, E, scale, resid, gap_rel);
    case 5: return launch_refine<5>(st, n, nk, H, Z, W1, W2, E, scale, resid, gap_rel);
    case 6: return launch_refine<6>(st, n, nk, H, Z, W1, W2, E, scale, resid, gap_rel);
    case 7: return launch_refine<7>(st, n, nk, H, Z, W1, W2, E, scale, resid, gap_rel);
    default: return launch_refine<8>(st, n, nk, H, Z, W1, W2, E, scale, resid, gap_rel);
  }
}

int col_set_smem_limits() {
  RTB_TRY(refine_limit<5>());
  RTB_TRY(refine_limit<6>());
  RTB_TRY(refine_limit<7>());
  RTB_TRY(refine_limit<8>());
  RTB_TRY((col_limits<kMul, kKubo>()));
  RTB_TRY((col_limits<kMulH, kStore>()));
  RTB_TRY((col_limits<kMul, kExact>()));
  RTB_TRY((col_limits<kMul, kImK>()));
  RTB_TRY((col_limits<kLoad, kAbs2>()));
  return RTB_OK;
}

}  // namespace rtb
