// The EnergyCut Fermi cut on the device: vertex Omega in tracked band order,
// then the zero-width cut of every (cell, simplex, band) for a list of
// chemical potentials (integrate_fermi_cut_2d_t0 / _3d_t0,
// src/response/energy_cut.rs:1231-1345, 1650-1797).  The per-simplex rules
// are energy_cut_core.hpp, the same code as the host part (energy_cut.cpp).
//
// One lane per (cell, simplex, band), lanes of a wave on consecutive bands.
// For each mu a lane settles the empty and full cases itself; the few that
// are cut (mu strictly inside the band's range on the simplex) are taken by
// the whole wave, two at a time for n <= 32: the 32 or 64 lanes of a group
// split the band sum over m of each quadrature point and add their shares in
// a fixed butterfly, so the loads of E and Im K rows are coalesced instead of
// one lane walking n bands.  The 64 lanes' contributions are then summed by
// DPP in a fixed order into a per-wave partial, and the partials are summed
// per mu in a fixed order (column_sums): the result does not depend on
// scheduling.
#include <limits>

#include "eigh.hpp"
#include "energy_cut_core.hpp"
#include "gpu_team.hpp"

namespace rtb {

namespace {

__global__ void cut_omega_kernel(cut::View V, size_t nk, double eta, double* __restrict__ om) {
  const size_t g = blockIdx.x * 256ull + threadIdx.x;
  if (g >= nk * static_cast<size_t>(V.n)) return;
  om[g] = cut::vertex_omega(V, g / V.n, static_cast<int>(g % V.n), eta);
}

// simplex s of a cell with band b, item g = (cell * S + s) * n + b
template <int DIM>
struct Simplex {
  static constexpr int NV = DIM + 1;
  size_t vs[NV];
  double c[NV][DIM];
  double e_v[NV], om_v[NV];
  double measure, scale;
  int b;
};

template <int DIM>
__device__ inline void load_simplex(const cut::View& V, const double* __restrict__ om, size_t g, size_t nx, size_t ny,
                                    size_t nz, Simplex<DIM>& x) {
  constexpr int S = DIM == 2 ? 4 : 5;  // simplices per cell
  const int n = V.n;
  const size_t cell = g / (static_cast<size_t>(S) * n);
  const int s = static_cast<int>((g / n) % S);
  x.b = static_cast<int>(g % n);
  if constexpr (DIM == 2) {
    cut::cell_triangle(cell / ny, cell % ny, nx, ny, s, x.vs, x.c);
    x.measure = cut::tri_area(x.c);
    const double half_vol = (1.0 / static_cast<double>(nx)) * (1.0 / static_cast<double>(ny)) / 4.0;
    x.scale = half_vol / x.measure;
  } else {
    double vol;
    cut::cell_tetrahedron(cell / (ny * nz), (cell / nz) % ny, cell % nz, nx, ny, nz, s, x.vs, x.c, &vol);
    x.measure = cut::tet_vol(x.c[0], x.c[1], x.c[2], x.c[3]);
    x.scale = vol / x.measure;
  }
  for (int q = 0; q < Simplex<DIM>::NV; ++q) {
    x.e_v[q] = cut::band(V, x.vs[q], x.b);
    x.om_v[q] = om[x.vs[q] * n + x.b];
  }
}

// Lane t's share of the band sum of eval_berry_band_at_lam_buf
// (kernel.rs:138-182): the terms m = t, t + G, ..; the G lanes' shares add up
// to the sum.  The lane's KM terms (E and Im K behind the tracking
// permutation) are gathered once per cut item, and every quadrature point of
// the item is evaluated from registers.
template <int NV, int KM>
struct CachedLaneBandSum {
  double eb[NV];
  double em[KM][NV], km[KM][NV];
  bool use[KM];
  double eta2;
  __device__ CachedLaneBandSum(const cut::View& M, const size_t* vs, int b, double eta, int t, int G) {
    eta2 = eta * eta;
#pragma unroll
    for (int v = 0; v < NV; ++v) eb[v] = cut::band(M, vs[v], b);
#pragma unroll
    for (int u = 0; u < KM; ++u) {
      const int m = t + G * u;
      use[u] = m < M.n && m != b;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        em[u][v] = use[u] ? cut::band(M, vs[v], m) : 0.0;
        km[u][v] = use[u] ? cut::kim(M, vs[v], b, m) : 0.0;
      }
    }
  }
  template <int NVV>
  __device__ double at(const double* lam) const {
    static_assert(NVV == NV, "vertex count");
    double en = 0.0;
#pragma unroll
    for (int v = 0; v < NV; ++v)
      if (lam[v] != 0.0) en += eb[v] * lam[v];
    double im = 0.0;
#pragma unroll
    for (int u = 0; u < KM; ++u) {
      if (!use[u]) continue;
      double e = 0.0, k = 0.0;
#pragma unroll
      for (int v = 0; v < NV; ++v)
        if (lam[v] != 0.0) e += em[u][v] * lam[v];
#pragma unroll
      for (int v = 0; v < NV; ++v)
        if (lam[v] != 0.0) k += km[u][v] * lam[v];
      const double de = en - e;
      const double denom = de * de + eta2;
      if (denom < 1e-30) continue;
      im += k / denom;
    }
    return -2.0 * im;
  }
};

// KM: terms per lane, ceil(n / G) with G = 32 lanes per item for n <= 32,
// 64 above.
template <int DIM, int KM>
__global__ void __launch_bounds__(256) cut_kernel(cut::View V, const double* __restrict__ om, size_t nx, size_t ny,
                                                  size_t nz, const double* __restrict__ mu, int n_mu, double eta,
                                                  double* __restrict__ partial) {
  constexpr int S = DIM == 2 ? 4 : 5;
  constexpr int NV = DIM + 1;
  const int n = V.n;
  const int G = n <= 32 ? 32 : 64;  // lanes per cut item
  const int lane = threadIdx.x & 63;
  const int t = lane & (G - 1);
  const size_t g = blockIdx.x * 256ull + threadIdx.x;
  const size_t g0 = g - lane;  // the wave's first item
  const size_t total = nx * ny * nz * S * static_cast<size_t>(n);
  bool live = g < total;
  Simplex<DIM> x{};
  double full_val = 0.0, e_min = 0.0, e_max = 0.0;
  if (live) {
    load_simplex<DIM>(V, om, g, nx, ny, nz, x);
    live = !(x.measure < cut::kEps);  // degenerate simplices of ragged meshes
    e_min = e_max = x.e_v[0];
    double osum = x.om_v[0];
    for (int q = 1; q < NV; ++q) {
      e_min = cut::dmin(e_min, x.e_v[q]);
      e_max = cut::dmax(e_max, x.e_v[q]);
      osum += x.om_v[q];
    }
    full_val = x.measure * osum / static_cast<double>(NV);
  }
  double* out = partial + (g / 64) * static_cast<size_t>(n_mu);
  for (int im = 0; im < n_mu; ++im) {
    const double m = mu[im];
    double v = 0.0;
    bool need = false;
    if (live) {
      // the partition points of the host loop: mu >= e_max - eps is the full
      // range, mu <= e_min + eps below it is empty, the rest is cut
      if (!(m < e_max - cut::kEps))
        v = x.scale * full_val;
      else
        need = !(m <= e_min + cut::kEps);
    }
    unsigned long long mask = __ballot(need);
    while (mask) {  // wave-uniform: every lane runs every pass
      const int l0 = __builtin_ctzll(mask);
      mask &= mask - 1;
      int l1 = -1;
      if (G == 32 && mask) {
        l1 = __builtin_ctzll(mask);
        mask &= mask - 1;
      }
      const int src = (G == 32 && lane >= 32) ? l1 : l0;  // this group's item
      double r = 0.0;
      if (src >= 0) {
        Simplex<DIM> y;
        load_simplex<DIM>(V, om, g0 + src, nx, ny, nz, y);
        const CachedLaneBandSum<NV, KM> f(V, y.vs, y.b, eta, t, G);
        const double one = t == 0 ? 1.0 : 0.0;
        if constexpr (DIM == 2)
          r = cut::hybrid_tri_by(y.c, y.e_v, y.om_v, m, f, one);
        else
          r = cut::hybrid_tet_by(y.c, y.e_v, y.om_v, m, f, one);
      }
      for (int o = G / 2; o > 0; o >>= 1) r += __shfl_xor(r, o);
      // group 0 (lanes 0..G-1) holds item l0's rule, group 1 item l1's; the
      // owners may sit in either half
      const double r0 = __shfl(r, 0), r1 = __shfl(r, 32);
      if (lane == l0) v = x.scale * r0;
      if (lane == l1) v = x.scale * r1;
    }
    v = wave_sum64(v);
    if (lane == 0) out[im] = v;
  }
}

// ---- many chemical potentials: lanes over mu ----
// With a grid of chemical potentials finer than the bands' spread over a
// simplex (the thermal convolution's: width / 10 apart) an item is cut at
// hundreds of them, and the kernel above gathers its vertex data and adds up
// a split band sum for each one.  Here a wave takes an item once: its lanes
// copy E and Im K of the simplex's vertices, in ascending order of the band's
// energy, to LDS and then take the item's sub-simplices of every chemical
// potential, one per lane (1, 3 or 1 of a tetrahedron with one, two or three
// vertices below mu, 1 or 2 of a triangle), each lane running the whole band
// sums of its quadrature points from broadcast LDS reads; up to 32 sub-simplices
// share the wave's lanes evenly, 2 to 32 for each one's band sum, added in a fixed
// butterfly (n = 32, 128 x 128, 256 mu over the band width: the call 12.2 ms with
// one lane each, 6.0 ms).  The sub-simplices
// of a mu are added in a fixed order, items follow each other in a fixed order
// within a wave, a wave's sums are per mu, and the full items enter as steps
// (one value at their first full mu, summed up at the end), so the result
// does not depend on scheduling.
// Bound: FP64 vector issue of the band sums.  20 x 18 x 16 cells of 5 simplices
// and 12 bands, 2985 chemical potentials: 7.7 ms (294 ms by the kernel above).
constexpr int kCutMu = 256;  // chemical potentials per wave (their sums sit in LDS), blocks of them in grid.y

// LDS of a wave (doubles): sums and steps per mu, a sub-simplex value each,
// then E and Im K [n][NV]
__host__ __device__ inline size_t cut_mu_wave_doubles(int n, int nv) {
  return static_cast<size_t>(2 + (nv - 1)) * kCutMu + 2 * static_cast<size_t>(n) * nv;
}

// The vertices of sub-simplex kind `kind` as sorted vertex pairs (p, q), four
// bits each (p | q << 2), vertex k at bits 4k: the point of edge p-q on the
// mu plane, or vertex p itself for p = q (clip_triangle, energy_cut.rs:1120-1169;
// tetrahedron_occupied_hybrid, energy_cut.rs:1529-1640, where kind 4 is the
// unoccupied corner).
__device__ constexpr unsigned sub_code(int p0, int q0, int p1, int q1, int p2, int q2, int p3, int q3) {
  return static_cast<unsigned>((p0 | q0 << 2) | (p1 | q1 << 2) << 4 | (p2 | q2 << 2) << 8 | (p3 | q3 << 2) << 12);
}
template <int NV>
__device__ inline unsigned sub_vertices(int kind) {
  if constexpr (NV == 4) {
    constexpr unsigned k0 = sub_code(0, 0, 0, 1, 0, 2, 0, 3), k1 = sub_code(0, 0, 1, 1, 0, 2, 1, 3),
                       k2 = sub_code(0, 0, 0, 2, 0, 3, 1, 3), k3 = sub_code(1, 1, 1, 2, 1, 3, 0, 2),
                       k4 = sub_code(3, 3, 0, 3, 1, 3, 2, 3);
    return kind == 0 ? k0 : (kind == 1 ? k1 : (kind == 2 ? k2 : (kind == 3 ? k3 : k4)));
  } else {
    constexpr unsigned k0 = sub_code(0, 0, 0, 1, 0, 2, 0, 0), k1 = sub_code(0, 0, 1, 1, 0, 2, 0, 0),
                       k2 = sub_code(1, 1, 0, 2, 1, 2, 0, 0);
    return kind == 0 ? k0 : (kind == 1 ? k1 : k2);
  }
}

template <int DIM>
__global__ void __launch_bounds__(256) cut_mu_kernel(cut::View V, const double* __restrict__ om, size_t nx, size_t ny,
                                                     size_t nz, const double* __restrict__ mu, int mu_all, double eta,
                                                     double* __restrict__ partial) {
  constexpr int S = DIM == 2 ? 4 : 5;
  constexpr int NV = DIM + 1;
  extern __shared__ double smem[];
  const int n = V.n;
  const int mu0 = blockIdx.y * kCutMu;
  const int n_mu = mu_all - mu0 < kCutMu ? mu_all - mu0 : kCutMu;
  mu += mu0;
  partial += mu0;  // rows of mu_all values
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double* acc = smem + wave * cut_mu_wave_doubles(n, NV);  // [kCutMu] cut items per mu
  double* step = acc + kCutMu;                             // [kCutMu] full items by their first full mu
  double* sub = step + kCutMu;                             // [DIM * kCutMu] the item's sub-simplices
  double* sE = sub + DIM * kCutMu;                         // [n][NV]
  double* sK = sE + n * NV;
  const size_t w = blockIdx.x * 4ull + wave, nw = gridDim.x * 4ull;
  const size_t total = nx * ny * nz * S * static_cast<size_t>(n);
  for (int i = lane; i < kCutMu; i += 64) {
    acc[i] = 0.0;
    step[i] = 0.0;
  }
  GpuTeam tm;
  tm.wave_sync();
  // first index in [a, b) with mu above x (or mu >= x when !above)
  const auto first = [&](int a, int b, double x, bool above) {
    while (a < b) {
      const int c = (a + b) / 2;
      const double m = mu[c];
      if (above ? m <= x : m < x)
        a = c + 1;
      else
        b = c;
    }
    return a;
  };
  const double eta2 = eta * eta;
  for (size_t g0 = w * 64; g0 < total; g0 += nw * 64) {
    // lane = item g0 + lane: its first cut and first full mu (the partition
    // points of the sorted mu: full from mu >= e_max - eps on, below that
    // empty up to mu <= e_min + eps, the rest cut)
    const size_t g = g0 + lane;
    int lo = n_mu, hi = n_mu;
    double full = 0.0;
    if (g < total) {
      Simplex<DIM> x;
      load_simplex<DIM>(V, om, g, nx, ny, nz, x);
      if (!(x.measure < cut::kEps)) {  // degenerate simplices of ragged meshes
        double e_min = x.e_v[0], e_max = x.e_v[0], osum = x.om_v[0];
        for (int q = 1; q < NV; ++q) {
          e_min = cut::dmin(e_min, x.e_v[q]);
          e_max = cut::dmax(e_max, x.e_v[q]);
          osum += x.om_v[q];
        }
        full = x.scale * (x.measure * osum / static_cast<double>(NV));
        hi = first(0, n_mu, e_max - cut::kEps, false);
        lo = first(0, hi, e_min + cut::kEps, true);
      }
    }
    // full items in item order
    unsigned long long fm = __ballot(hi < n_mu);
    while (fm) {
      const int l = __builtin_ctzll(fm);
      fm &= fm - 1;
      const int h = __builtin_amdgcn_readlane(hi, l);
      const double f = lane_value(full, l);
      if (lane == 0) step[h] += f;
    }
    // cut items in item order
    unsigned long long cm = __ballot(lo < hi);
    while (cm) {
      const int l = __builtin_ctzll(cm);
      cm &= cm - 1;
      const int a0 = __builtin_amdgcn_readlane(lo, l), a1 = __builtin_amdgcn_readlane(hi, l);
      const double vfull = lane_value(full, l);
      Simplex<DIM> y;
      load_simplex<DIM>(V, om, g0 + l, nx, ny, nz, y);
      // vertices by ascending energy, ties in vertex order (sort_idx)
      size_t vs[NV];
      double e[NV];
#pragma unroll
      for (int q = 0; q < NV; ++q) {
        vs[q] = y.vs[q];
        e[q] = y.e_v[q];
      }
#pragma unroll
      for (int round = 0; round < NV; ++round)
#pragma unroll
        for (int i = round % 2; i + 1 < NV; i += 2)
          if (e[i + 1] < e[i]) {
            const double te = e[i];
            e[i] = e[i + 1];
            e[i + 1] = te;
            const size_t tv = vs[i];
            vs[i] = vs[i + 1];
            vs[i + 1] = tv;
          }
      tm.wave_sync();  // the previous item's reads are done
      for (int q = lane; q < n * NV; q += 64) {
        const int m = q / NV, v = q - m * NV;
        size_t vq = vs[0];
#pragma unroll
        for (int u = 1; u < NV; ++u) vq = u == v ? vs[u] : vq;
        sE[q] = cut::band(V, vq, m);
        sK[q] = cut::kim(V, vq, y.b, m);
      }
      tm.wave_sync();
      const double measure = y.measure;
      // units: one sub-simplex for the mu up to vertex 1's energy (i1), DIM of
      // them up to the next (i2; in 2D the rest), one above
      const int i1 = first(a0, a1, e[1] + cut::kEps, true);
      const int i2 = DIM == 3 ? first(i1, a1, e[DIM - 1] + cut::kEps, true) : a1;
      const int n1 = i1 - a0, n2 = i2 - i1;
      const int units = n1 + DIM * n2 + (a1 - i2);
      // few units: `parts` lanes (a power of two) split each one's band sum
      int sh = 0;
      while (sh < 5 && units << (sh + 1) <= 64) ++sh;
      const int parts = 1 << sh;
      for (int q = lane; q < units << sh; q += 64) {
        const int u = q >> sh;
        int i, kind;
        if (u < n1) {
          i = a0 + u;
          kind = 0;
        } else if (u < n1 + DIM * n2) {
          const int r = u - n1;
          i = i1 + r / DIM;
          kind = 1 + r % DIM;
        } else {
          i = i2 + (u - n1 - DIM * n2);
          kind = 4;
        }
        const double m = mu[i];
        const unsigned code = sub_vertices<NV>(kind);
        double sb[NV][NV];  // barycentric vertices
        double vol = measure;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
          const int p = (code >> (4 * k)) & 3, q = (code >> (4 * k + 2)) & 3;
          const double ep = cut::pick<NV>(e, p), de = cut::pick<NV>(e, q) - ep;
          double t = 0.5;
          if (!(fabs(de) < cut::kEps)) {
            t = (m - ep) / de;
            t = t < 0.0 ? 0.0 : (t > 1.0 ? 1.0 : t);
          }
          if (p == q) t = 0.0;
#pragma unroll
          for (int d = 0; d < NV; ++d) sb[k][d] = p == d ? 1.0 - t : (q == d ? t : 0.0);
          // |det| of the barycentric rows: the product of the edge vertices'
          // weights at the vertex no other row of the kind has
          if (p != q) {
            const bool one_minus = DIM == 3 ? kind == 4 || (kind >= 2 && k == 3) : kind == 2 && k == 1;
            vol *= one_minus ? 1.0 - t : t;
          }
        }
        double val = 0.0;
        if (!(vol < 1e-30)) {
          // the degree-2 rule: lam_k = wb sum of the vertices + (wa - wb) vertex k
          constexpr double wa = DIM == 3 ? cut::kTA : 2.0 / 3.0, wb = DIM == 3 ? cut::kTB : 1.0 / 6.0;
          double lam[NV][NV], en[NV], im[NV];
#pragma unroll
          for (int d = 0; d < NV; ++d) {
            double t = sb[0][d];
#pragma unroll
            for (int k = 1; k < NV; ++k) t += sb[k][d];
            t *= wb;
#pragma unroll
            for (int k = 0; k < NV; ++k) lam[k][d] = fma(wa - wb, sb[k][d], t);
          }
#pragma unroll
          for (int k = 0; k < NV; ++k) {
            im[k] = 0.0;
            en[k] = 0.0;
#pragma unroll
            for (int d = 0; d < NV; ++d) en[k] = fma(sE[y.b * NV + d], lam[k][d], en[k]);
          }
          const auto terms = [&](int first_mb, int step_mb) {
            for (int mb = first_mb; mb < n; mb += step_mb) {
              if (mb == y.b) continue;
              double ev[NV], kv[NV];
#pragma unroll
              for (int d = 0; d < NV; ++d) {
                ev[d] = sE[mb * NV + d];
                kv[d] = sK[mb * NV + d];
              }
#pragma unroll
              for (int k = 0; k < NV; ++k) {
                double de = en[k], kk = 0.0;
#pragma unroll
                for (int d = 0; d < NV; ++d) {
                  de = fma(-ev[d], lam[k][d], de);
                  kk = fma(kv[d], lam[k][d], kk);
                }
                const double denom = fma(de, de, eta2);
                // hardware reciprocal and two Newton steps; a division where
                // those would leave the number range
                double r = __builtin_amdgcn_rcp(denom);
                r = fma(r, fma(-denom, r, 1.0), r);
                r = fma(r, fma(-denom, r, 1.0), r);
                if (!(denom < 1e300)) r = 1.0 / denom;
                if (!(denom < 1e-30)) im[k] = fma(kk, r, im[k]);
              }
            }
          };
          if (sh == 0)
            terms(0, 1);  // one band at a time in the whole wave
          else
            terms(q & (parts - 1), parts);
          // the lanes of a unit hold the same vol and take the same branch
          for (int o = parts / 2; o > 0; o >>= 1)
#pragma unroll
            for (int k = 0; k < NV; ++k) im[k] += __shfl_xor(im[k], o);
          constexpr double wq = 1.0 / NV;
#pragma unroll
          for (int k = 0; k < NV; ++k) val += vol * wq * (-2.0 * im[k]);
        }
        if ((q & (parts - 1)) == 0) sub[u] = kind == 4 ? -val : val;
      }
      tm.wave_sync();
      // the sub-simplices of each mu, in order
      for (int i = a0 + lane; i < a1; i += 64) {
        double r;
        if (i < i1) {
          r = sub[i - a0];
        } else if (i < i2) {
          const int u = n1 + DIM * (i - i1);
          r = sub[u];
#pragma unroll
          for (int q = 1; q < DIM; ++q) r += sub[u + q];
        } else {
          r = sub[n1 + DIM * n2 + (i - i2)];
        }
        r *= y.scale;
        if (i >= i2) r += vfull;  // the full simplex minus the corner above mu
        acc[i] += r;
      }
    }
  }
  tm.wave_sync();
  // out[i] = cut sums + the steps up to i, 64 at a time with a carry
  double carry = 0.0;
  for (int i0 = 0; i0 < n_mu; i0 += 64) {
    const int i = i0 + lane;
    double s = i < n_mu ? step[i] : 0.0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const double t = __shfl_up(s, o);
      if (lane >= o) s += t;
    }
    s += carry;
    if (i < n_mu) partial[w * mu_all + i] = acc[i] + s;
    carry = lane_value(s, 63);
  }
}

// ---- band tracking (global_band_track, tracking.rs:123-163) ----
// One workgroup per vertex of a level: the squared overlaps of its scheduled
// neighbours (rows in the neighbour's tracked order) summed in neighbour
// order and divided by their count into M, as the host walk forms them;
// then greedy_assign (tracking.rs:44-68): rows by descending row maximum
// (stable), each taking its largest unassigned column, the lowest column
// among equal values.  Where all rows' best columns differ each row takes its
// own; otherwise the rows are ranked and wave 0 walks only those whose best
// column is taken when their turn comes, each scanning the free columns.  The
// same operations on the same values as the host walk, so the permutations
// are identical.  M [n][n] sits in LDS up to kTrackLdsMaxN bands and above in
// a global slice per workgroup of the launch (n = 256: 512 KiB); there a wave
// builds each row and ranks its first kTrackTop columns in registers, a row
// whose best column is taken takes the first free one of them, and only when
// all are taken does wave 0 scan the row in global memory.
// Bound: a chain of launches, one per level (4.3 us each where they do next to
// nothing, n = 4); in one, the latencies of schedule, permutations and overlaps
// in turn.  Per level, 2D: n = 32 14.8 -> 7.7 us, n = 64 32 -> 15, n = 128
// 89 -> 43, n = 160 136 -> 101 against a thread per row's maximum and a walk of
// every row.
constexpr int kTrackMaxDep = 6;  // visited neighbours of a 3D vertex at most
static_assert(sizeof(TrackEntry) == 8 * sizeof(unsigned), "schedule entry layout");
static_assert(kTrackDevMaxN <= 256, "the greedy's assigned-column mask is four 64-bit words");

// LDS bytes: M when it is in LDS, then rmax [n], best/order/bsort/owner [n] each,
// the neighbours' permutations [kTrackMaxDep][n] and, with M in global
// memory, each row's first kTrackTop columns [n][kTrackTop]
constexpr int kTrackTop = 4;
size_t track_smem(int n) {
  const bool lds = n <= kTrackLdsMaxN;
  const size_t m = lds ? static_cast<size_t>(n) * n * sizeof(double) : 0;
  return m + n * sizeof(double) + (4 + kTrackMaxDep + (lds ? 0 : kTrackTop)) * static_cast<size_t>(n) * sizeof(int);
}

__global__ void identity_perm_kernel(size_t total, int n, int* __restrict__ perm) {
  const size_t g = blockIdx.x * 256ull + threadIdx.x;
  if (g < total) perm[g] = static_cast<int>(g % n);
}

// The overlap sum over the neighbours divided by their count: x / 1, x * 0.5
// and x * 0.25 are the correctly rounded x / c for c = 1, 2, 4 (exact
// scalings), so only 3, 5 and 6 take the division.
__device__ inline double by_count(double x, int cnt, double dc) {
  return cnt == 1 ? x : (cnt == 2 ? x * 0.5 : (cnt == 4 ? x * 0.25 : x / dc));
}

// Threads per vertex: the build waits on loads, and a level holds few vertices,
// so as many rows at once as fit (n = 32, 128 x 128: 3.63 ms with 256 threads,
// 2.95 with 512, 2.63 with 1024; n <= 16 the same within 4%); with M in global
// memory one row per wave in flight.
constexpr int kTrackThreads = 1024;
constexpr int kTrackThreadsWide = 1024;
template <bool kLdsM>
__global__ void __launch_bounds__(kLdsM ? kTrackThreads : kTrackThreadsWide) track_kernel(const double* __restrict__ ovx, const double* __restrict__ ovy,
                                                   const double* __restrict__ ovz, size_t ny, size_t nz, int n,
                                                   const TrackEntry* __restrict__ sched, double* __restrict__ mwork,
                                                   int* __restrict__ perm) {
  constexpr int NT = kLdsM ? kTrackThreads : kTrackThreadsWide;
  extern __shared__ double smem[];
  const int nn = n * n;
  const size_t n2 = static_cast<size_t>(nn);
  double* M = kLdsM ? smem : mwork + blockIdx.x * n2;  // [n][n]
  double* rmax = kLdsM ? smem + n2 : smem;               // [n]
  int* best = reinterpret_cast<int*>(rmax + n);          // [n] each row's best column over all columns
  int* order = best + n;                                 // [n] rows by descending maximum
  int* bsort = order + n;                                // [n] best[order[s]]
  int* owner = bsort + n;                                // [n] a column's first rank
  int* pv = owner + n;                                   // [kTrackMaxDep][n] the neighbours' permutations
  int* top = pv + kTrackMaxDep * n;                      // [n][kTrackTop] (M in global memory only)
  const TrackEntry te = sched[blockIdx.x];              // uniform: one scalar load
  const size_t nb = te.v;
  const int cnt = static_cast<int>(te.cnt);
  if (cnt == 0) return;  // vertex 0 keeps the identity
  const int tid = threadIdx.x;
  __shared__ unsigned long long claimed[kTrackDevMaxN / 64];  // columns that are some row's best
  if (tid < kTrackDevMaxN / 64) claimed[tid] = 0;
  for (int a = tid; a < n; a += NT) owner[a] = n;
#pragma unroll
  for (int r = 0; r < kTrackMaxDep; ++r)
    if (r < cnt)
      for (int a = tid; a < n; a += NT) pv[r * n + a] = perm[static_cast<size_t>(te.dep[r]) * n + a];
  // each neighbour's overlap block and orientation; the pair's axis from its
  // index step, x first (with ny = 1 the x and y steps coincide and only x
  // pairs exist)
  const double* base[kTrackMaxDep];
  bool lower[kTrackMaxDep];  // nb is the pair's lower vertex: its raw band is the row
#pragma unroll
  for (int r = 0; r < kTrackMaxDep; ++r) {
    base[r] = nullptr;
    lower[r] = false;
    if (r < cnt) {
      const size_t vn = te.dep[r];
      const size_t lo = nb < vn ? nb : vn, step = (nb < vn ? vn : nb) - lo;
      const double* axis = step == ny * nz ? ovx : (step == nz ? ovy : ovz);
      base[r] = axis + lo * n2;
      lower[r] = nb == lo;
    }
  }
  __syncthreads();
  const double dc = static_cast<double>(cnt);
  // entry (a, b) of M: the neighbours' values in neighbour order
  const auto entry = [&](int a, int b) {
    double x = 0.0;
#pragma unroll
    for (int r = 0; r < kTrackMaxDep; ++r) {
      if (r < cnt) {
        const size_t pa = static_cast<size_t>(pv[r * n + a]);
        const double y = lower[r] ? base[r][static_cast<size_t>(b) * n + pa] : base[r][pa * n + b];
        x = r == 0 ? y : x + y;
      }
    }
    return by_count(x, cnt, dc);
  };
  if constexpr (kLdsM) {
    // a row per group of sw lanes (16, 32 or a wave, the least that holds it
    // or 64): built, stored and its maximum (NaN never ranked) and best
    // column, the lowest among equal values, merged over the group
    const int sw = n <= 16 ? 16 : (n <= 32 ? 32 : 64);
    for (int a = tid / sw; a < n; a += NT / sw) {
      double bv = -1.0;
      int bj = 0;
      for (int b = tid % sw; b < n; b += sw) {
        const double x = entry(a, b);
        M[a * n + b] = x;
        if (x > bv) {
          bv = x;
          bj = b;
        }
      }
      for (int o = sw / 2; o > 0; o >>= 1) {
        const double ov = __shfl_xor(bv, o);
        const int oj = __shfl_xor(bj, o);
        if (ov > bv || (ov == bv && oj < bj)) {
          bv = ov;
          bj = oj;
        }
      }
      if (tid % sw == 0) {
        rmax[a] = bv;
        best[a] = bj;
        atomicOr(&claimed[bj >> 6], 1ull << (bj & 63));
      }
    }
  } else {
    // a row per wave, each lane its columns b = lane + 64 c: the row is
    // built, stored, and ranked from registers.  The columns in the order
    // of the host scan (larger value first, then lower column; NaN never
    // ranked) are found kTrackTop times over, each round among the columns
    // after the previous round's; the lanes' (value, column) pairs merge by
    // that order, and a lane or row with no candidate gives (-1, 0), which
    // every candidate (>= 0) beats.  Round 0 is the row's maximum and best
    // column as the host scan gives them.
    const int wv = tid >> 6, ln = tid & 63;
    for (int a = wv; a < n; a += NT / 64) {
      double xv[kTrackDevMaxN / 64];
#pragma unroll
      for (int c = 0; c < kTrackDevMaxN / 64; ++c) {
        const int b = ln + 64 * c;
        xv[c] = __builtin_nan("");
        if (b < n) {
          xv[c] = entry(a, b);
          M[static_cast<size_t>(a) * n + b] = xv[c];
        }
      }
      double pvl = 0.0;
      int pcl = -1;
#pragma unroll
      for (int k = 0; k < kTrackTop; ++k) {
        double bv = -1.0;
        int bj = 0;
#pragma unroll
        for (int c = 0; c < kTrackDevMaxN / 64; ++c) {
          const double x = xv[c];
          const int b = ln + 64 * c;
          const bool after = k == 0 || x < pvl || (x == pvl && b > pcl);
          if (after && x > bv) {
            bv = x;
            bj = b;
          }
        }
        for (int o = 32; o > 0; o >>= 1) {
          const double ov = __shfl_xor(bv, o);
          const int oj = __shfl_xor(bj, o);
          if (ov > bv || (ov == bv && oj < bj)) {
            bv = ov;
            bj = oj;
          }
        }
        if (ln == 0) {
          if (k == 0) {
            rmax[a] = bv;
            best[a] = bj;
            atomicOr(&claimed[bj >> 6], 1ull << (bj & 63));
          }
          top[a * kTrackTop + k] = bv >= 0.0 ? bj : -1;  // -1: no further candidate
        }
        pvl = bv;
        pcl = bj;
      }
    }
  }
  __syncthreads();
  int* out = perm + nb * n;
  // where no column is the best of two rows each row takes its own, whatever
  // the order
  int distinct = 0;
  for (int c = 0; c < kTrackDevMaxN / 64; ++c) distinct += __popcll(claimed[c]);
  if (distinct == n) {
    for (int i = tid; i < n; i += NT) out[i] = best[i];
    return;
  }
  // the stable descending sort as ranks; owner: the first rank a column is
  // the best of
  for (int i = tid; i < n; i += NT) {
    const double x = rmax[i];
    int rank = 0;
#pragma unroll 8
    for (int k = 0; k < n; ++k) {
      const double y = rmax[k];
      rank += (y > x || (y == x && k < i)) ? 1 : 0;
    }
    order[rank] = i;
    bsort[rank] = best[i];
    atomicMin(&owner[best[i]], rank);
  }
  __syncthreads();
  if (tid >= 64) return;
  const int lane = tid;
  // Ranks that do not get their best column, 64 c .. 64 c + 63 in word c (the
  // same in every lane): those whose column has an earlier owner and, as the
  // walk finds them, those whose column a displaced row before them takes.
  // At rank s a column is taken if its owner comes before s (the owner has it
  // or found it taken) or a displaced row took it; bits: the latter's columns.
  constexpr int NW = kLdsM ? kTrackLdsMaxN / 64 : kTrackDevMaxN / 64;
  unsigned long long late[NW], bits[NW];
  int own[NW];  // of columns lane + 64 c
#pragma unroll
  for (int c = 0; c < NW; ++c) {
    const int s = lane + 64 * c;
    late[c] = __ballot(s < n && owner[s < n ? bsort[s] : 0] != s);
    bits[c] = 0;
    own[c] = s < n ? owner[s] : 0;
  }
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    while (late[w]) {
      const int q = __ffsll(late[w]) - 1, s = 64 * w + q;
      late[w] &= late[w] - 1;
      const int r = order[s];
      int j = -1;
      if constexpr (!kLdsM) {
        // the first free column of the row's ranked list (entry 0 is its best)
        // is the free columns' maximum; the full scan only when the list runs
        // out
#pragma unroll
        for (int k = 1; k < kTrackTop; ++k) {
          const int c = top[r * kTrackTop + k];
          if (c < 0) break;
          bool t = owner[c] < s;
#pragma unroll
          for (int v = 0; v < NW; ++v) t = t || (v == c >> 6 && ((bits[v] >> (c & 63)) & 1ull));
          if (!t) {
            j = c;
            break;
          }
        }
      }
      if (j < 0) {  // the scan over the free columns
        // no candidate: (-1, 0), as the host scan's start; every real
        // candidate is >= 0 and NaN never wins
        double bv = -1.0;
        int bj = 0;
#pragma unroll
        for (int c = 0; c < NW; ++c) {
          const int jj = lane + 64 * c;
          if (jj < n) {
            const double v = M[static_cast<size_t>(r) * n + jj];
            if (!(own[c] < s || ((bits[c] >> lane) & 1ull)) && v > bv) {
              bv = v;
              bj = jj;
            }
          }
        }
        for (int o = 32; o > 0; o >>= 1) {
          const double ov = __shfl_xor(bv, o);
          const int oj = __shfl_xor(bj, o);
          if (ov > bv || (ov == bv && oj < bj)) {
            bv = ov;
            bj = oj;
          }
        }
        j = __builtin_amdgcn_readfirstlane(bj);
      }
      const int oj = owner[j];  // n: no row's best
#pragma unroll
      for (int c = 0; c < NW; ++c) {
        if (j >> 6 == c) bits[c] |= 1ull << (j & 63);
        if (oj > s && oj < n && oj >> 6 == c) late[c] |= 1ull << (oj & 63);
      }
      if (lane == 0) bsort[s] = j;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // bsort as lane 0 left it
#pragma unroll
  for (int c = 0; c < NW; ++c) {
    const int s = lane + 64 * c;
    if (s < n) out[order[s]] = bsort[s];
  }
}

}  // namespace

int energy_cut_omega(hipStream_t st, int n, size_t nk, const double* E, const double* Ki, const int* perm, double eta,
                     double* om) {
  const size_t total = nk * static_cast<size_t>(n);
  if (total == 0) return RTB_OK;
  const cut::View V{n, E, Ki, 1, perm};
  hipLaunchKernelGGL(cut_omega_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, st, V, nk,
                     eta, om);
  RTB_HIP(hipGetLastError());
  return RTB_OK;
}

static size_t energy_cut_waves(int dim, size_t nx, size_t ny, size_t nz, int n) {
  const size_t total = nx * ny * nz * (dim == 2 ? 4 : 5) * static_cast<size_t>(n);
  return (total + 255) / 256 * 4;
}

// Lanes over mu (cut_mu_kernel) from 64 chemical potentials on.  Whole calls, split
// band sum against lanes over mu, for windows of 0.05, 1 and 30 band widths, in ms:
//   2D n = 32, 128 x 128    64 mu  5.36/4.72  4.87/4.97  4.54/4.47
//                          256 mu  8.36/5.18  6.39/6.01  5.19/4.69
//   2D n = 4, 200 x 200     64 mu  3.38/3.16  3.23/3.29  3.10/3.11
//   2D n = 96, 24 x 24      64 mu  10.6/5.82  6.74/5.26  4.39/4.38
//   3D n = 12, 20 x 18 x 16 64 mu  9.57/1.49  4.65/1.86  1.13/1.09
// With fewer the split band sum is up to 5% ahead where an item is cut once or not at
// all (n = 12, 20 x 18 x 16, 4 mu 1.40/1.11  1.07/1.12  0.89/0.91), the lanes over mu in
// narrow windows only.
static bool lanes_over_mu(size_t n_mu) { return n_mu >= 64; }
// partial rows (waves); with lanes over mu a wave covers one or more groups of
// 64 items, so that the rows stay few
constexpr size_t kCutMuRows = 8192;
size_t energy_cut_rows(int dim, size_t nx, size_t ny, size_t nz, int n, size_t n_mu) {
  const size_t waves = energy_cut_waves(dim, nx, ny, nz, n);
  return lanes_over_mu(n_mu) ? std::min(waves, kCutMuRows) : waves;
}

namespace {

template <int DIM>
int launch_cut_dim(hipStream_t st, int n, unsigned blocks, const cut::View& V, const double* om, size_t nx, size_t ny,
                   size_t nz, const double* mu, int c, double eta, double* partial) {
  // the kernel's lanes per item: 32 for n <= 32, else 64; KM = ceil(n / G)
  const int G = n <= 32 ? 32 : 64;
  const int km = (n + G - 1) / G;
  if (km <= 1)
    hipLaunchKernelGGL((cut_kernel<DIM, 1>), dim3(blocks), dim3(256), 0, st, V, om, nx, ny, nz, mu, c, eta, partial);
  else if (km == 2)
    hipLaunchKernelGGL((cut_kernel<DIM, 2>), dim3(blocks), dim3(256), 0, st, V, om, nx, ny, nz, mu, c, eta, partial);
  else if (km <= 4)
    hipLaunchKernelGGL((cut_kernel<DIM, 4>), dim3(blocks), dim3(256), 0, st, V, om, nx, ny, nz, mu, c, eta, partial);
  else
    return fail(RTB_ERR_UNSUPPORTED, "the Fermi cut is for n <= 256");
  RTB_HIP(hipGetLastError());
  return RTB_OK;
}

int launch_cut(hipStream_t st, int dim, int n, unsigned blocks, const cut::View& V, const double* om, size_t nx,
               size_t ny, size_t nz, const double* mu, int c, double eta, double* partial) {
  if (dim == 2) return launch_cut_dim<2>(st, n, blocks, V, om, nx, ny, nz, mu, c, eta, partial);
  return launch_cut_dim<3>(st, n, blocks, V, om, nx, ny, nz, mu, c, eta, partial);
}

}  // namespace

int energy_cut_t0(hipStream_t st, int dim, size_t nx, size_t ny, size_t nz, int n, const double* E, const double* Ki,
                  const int* perm, const double* om, const double* mu, size_t n_mu, double eta, double* partial,
                  size_t chunk, double* out) {
  if (dim != 2 && dim != 3) return fail(RTB_ERR_INVALID_DIMENSION, "the cut is for 2D and 3D meshes");
  if (chunk == 0) return fail(RTB_ERR_INVALID_ARGUMENT, "zero mu chunk");
  const size_t waves = energy_cut_waves(dim, nx, ny, nz, n);
  const unsigned blocks = static_cast<unsigned>(waves / 4);
  const cut::View V{n, E, Ki, 1, perm};
  if (lanes_over_mu(n_mu)) {
    const size_t rows = energy_cut_rows(dim, nx, ny, nz, n, n_mu);
    const size_t smem = 4 * cut_mu_wave_doubles(n, dim + 1) * sizeof(double);
    for (size_t m0 = 0; m0 < n_mu; m0 += chunk) {
      const int c = static_cast<int>(std::min(chunk, n_mu - m0));
      const dim3 grid(static_cast<unsigned>(rows / 4), static_cast<unsigned>((c + kCutMu - 1) / kCutMu));
      if (dim == 2)
        hipLaunchKernelGGL(cut_mu_kernel<2>, grid, dim3(256), smem, st, V, om, nx, ny, nz, mu + m0, c, eta, partial);
      else
        hipLaunchKernelGGL(cut_mu_kernel<3>, grid, dim3(256), smem, st, V, om, nx, ny, nz, mu + m0, c, eta, partial);
      RTB_HIP(hipGetLastError());
      RTB_TRY(column_sums(st, partial, rows, c, out + m0));
    }
    return RTB_OK;
  }
  for (size_t m0 = 0; m0 < n_mu; m0 += chunk) {
    const int c = static_cast<int>(std::min(chunk, n_mu - m0));
    RTB_TRY(launch_cut(st, dim, n, blocks, V, om, nx, ny, nz, mu + m0, c, eta, partial));
    RTB_TRY(column_sums(st, partial, waves, c, out + m0));
  }
  return RTB_OK;
}

int energy_cut_track_smem_limits() {
  RTB_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&cut_mu_kernel<2>),
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              static_cast<int>(4 * cut_mu_wave_doubles(kTrackDevMaxN, 3) * sizeof(double))));
  RTB_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&cut_mu_kernel<3>),
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              static_cast<int>(4 * cut_mu_wave_doubles(kTrackDevMaxN, 4) * sizeof(double))));
  RTB_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&track_kernel<true>),
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              static_cast<int>(track_smem(kTrackLdsMaxN))));
  return RTB_OK;
}

int energy_cut_track_dev(hipStream_t st, size_t nx, size_t ny, size_t nz, int n, const double* ovx,
                         const double* ovy, const double* ovz, const TrackEntry* sched,
                         const std::vector<size_t>& level_start, double* mwork, size_t mwork_blocks, int* perm) {
  if (n < 1 || n > kTrackDevMaxN) return fail(RTB_ERR_UNSUPPORTED, "device band tracking is for n <= 256");
  const bool lds = n <= kTrackLdsMaxN;
  if (!lds && (!mwork || mwork_blocks == 0))
    return fail(RTB_ERR_INVALID_ARGUMENT, "device band tracking above 128 bands needs its matrix workspace");
  const size_t nk = nx * ny * nz;
  if (nk == 0) return RTB_OK;
  const size_t total = nk * static_cast<size_t>(n);
  hipLaunchKernelGGL(identity_perm_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, st, total,
                     n, perm);
  RTB_HIP(hipGetLastError());
  // level 0 is vertex 0 alone (no neighbours visited before it); above
  // kTrackLdsMaxN a level goes in launches of at most mwork_blocks vertices,
  // one workspace slice each
  const size_t step = lds ? std::numeric_limits<unsigned>::max() : mwork_blocks;
  for (size_t l = 1; l + 1 < level_start.size(); ++l) {
    for (size_t a = level_start[l]; a < level_start[l + 1]; a += step) {
      const size_t b = std::min(level_start[l + 1], a + step);
      if (lds)
        hipLaunchKernelGGL(track_kernel<true>, dim3(static_cast<unsigned>(b - a)), dim3(kTrackThreads), track_smem(n),
                           st, ovx, ovy, ovz, ny, nz, n, sched + a, nullptr, perm);
      else
        hipLaunchKernelGGL(track_kernel<false>, dim3(static_cast<unsigned>(b - a)), dim3(kTrackThreadsWide),
                           track_smem(n), st, ovx, ovy, ovz, ny, nz, n, sched + a, mwork, perm);
      RTB_HIP(hipGetLastError());
    }
  }
  return RTB_OK;
}

}  // namespace rtb
