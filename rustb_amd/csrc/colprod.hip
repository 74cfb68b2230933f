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
// device).
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

template <int NT, int OP, int EP>
__global__ void __launch_bounds__(64 * NT) __attribute__((amdgpu_waves_per_eu(2))) col_product_kernel(ColArgs a) {
  using Sh = ColShape<NT>;
  constexpr int RT = Sh::RT, NH = Sh::NH, TH = Sh::threads, N = 16 * NT;
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
    constexpr int EL = (16 * RT * kCK + TH - 1) / TH;  // staged elements per thread
    const int nc = (n + kCK - 1) / kCK;
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      const int r0 = 16 * RT * h;
      double2 px[EL], pb[4];
      auto load = [&](int k0) {
#pragma unroll
        for (int u = 0; u < EL; ++u) {
          const int q = tid + TH * u;
          double2 x = make_double2(0.0, 0.0);
          if (16 * RT * kCK % TH == 0 || q < 16 * RT * kCK) {
            if constexpr (OP == kMul) {  // lanes along k within a row
              const int i = r0 + q / kCK, k = k0 + q % kCK;
              if (i < n && k < n) x = X[static_cast<unsigned>(i * n + k)];
            } else {  // X^H: lanes along the row of X
              const int k = k0 + q / (16 * RT), i = r0 + q % (16 * RT);
              if (i < n && k < n) x = X[static_cast<unsigned>(k * n + i)];
            }
          }
          px[u] = x;
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int k = k0 + 4 * s + fk;
          pb[s] = k < n && col < n ? Z[static_cast<unsigned>(k * n + col)] : make_double2(0.0, 0.0);
        }
      };
      d4 a1[RT], a2[RT], a3[RT];
#pragma unroll
      for (int t = 0; t < RT; ++t) a1[t] = a2[t] = a3[t] = d4{0.0, 0.0, 0.0, 0.0};
      load(0);
      if (h > 0) __syncthreads();  // the previous group's last chunk is consumed
      for (int c = 0; c < nc; ++c) {
        double* b = smem + (c & 1) * Sh::p1;
#pragma unroll
        for (int u = 0; u < EL; ++u) {
          const int q = tid + TH * u;
          if (16 * RT * kCK % TH == 0 || q < 16 * RT * kCK) {
            const int i = OP == kMul ? q / kCK : q % (16 * RT), k = OP == kMul ? q % kCK : q / (16 * RT);
            const double re = px[u].x, im = OP == kMul ? px[u].y : -px[u].y;
            b[i * kCLd + k] = re;
            b[16 * RT * kCLd + i * kCLd + k] = im;
            b[2 * 16 * RT * kCLd + i * kCLd + k] = re + im;
          }
        }
        double br[4], bi[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          br[s] = pb[s].x;
          bi[s] = pb[s].y;
        }
        __syncthreads();
        if (c + 1 < nc) load((c + 1) * kCK);  // in flight during the MFMAs
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const double bs = br[s] + bi[s];
          const double* f = b + fr * kCLd + 4 * s + fk;
#pragma unroll
          for (int t = 0; t < RT; ++t) {
            if (RT * h + t < NT) {
              const double* g = f + 16 * t * kCLd;
              a1[t] = mfma64(g[0], br[s], a1[t]);
              a2[t] = mfma64(g[16 * RT * kCLd], bi[s], a2[t]);
              a3[t] = mfma64(g[2 * 16 * RT * kCLd], bs, a3[t]);
            }
          }
          __builtin_amdgcn_sched_barrier(0);  // bounded look-ahead of the LDS reads (registers)
        }
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
  // ---- C_IJ = Z_I^H T_J, row tile by row tile ----
  constexpr int EL2 = 16 * N / TH;  // 4
  double2 pz[EL2];
  auto load2 = [&](int I) {
#pragma unroll
    for (int u = 0; u < EL2; ++u) {
      const int q = tid + TH * u;
      const int k = q / 16, c = 16 * I + q % 16;
      pz[u] = k < n && c < n ? Z[static_cast<unsigned>(k * n + c)] : make_double2(0.0, 0.0);
    }
  };
  double colsum = 0.0, colsum2 = 0.0;  // Omega (column sum of Q), metric
  load2(0);
  __syncthreads();  // the first product's buffers are free; sE, sS are visible
  const double Ej = sE[col], sj = sS[col];
#pragma unroll 1
  for (int I = 0; I < NT; ++I) {
    double* b = smem + (I & 1) * Sh::p2;
#pragma unroll
    for (int u = 0; u < EL2; ++u) {
      const int q = tid + TH * u;
      const double re = pz[u].x, im = -pz[u].y;  // Z^H
      b[q] = re;
      b[16 * N + q] = im;
      b[2 * 16 * N + q] = re + im;
    }
    __syncthreads();
    if (I + 1 < NT) load2(I + 1);
    double2 pp[4];
    if constexpr (EP == kExact || EP == kImK) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * I + 4 * r + fk;
        pp[r] = i < n && col < n ? P[static_cast<unsigned>(i * n + col)] : make_double2(0.0, 0.0);
      }
    }
    d4 c1 = {0.0, 0.0, 0.0, 0.0}, c2 = c1, c3 = c1;
#pragma unroll
    for (int K = 0; K < NT; ++K) {
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

int col_set_smem_limits() {
  RTB_TRY((col_limits<kMul, kKubo>()));
  RTB_TRY((col_limits<kMulH, kStore>()));
  RTB_TRY((col_limits<kMul, kExact>()));
  RTB_TRY((col_limits<kMul, kImK>()));
  RTB_TRY((col_limits<kLoad, kAbs2>()));
  return RTB_OK;
}

}  // namespace rtb
