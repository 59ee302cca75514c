// Mass-weighted Hessian spectrum of the non-frozen atoms (the rate prefactor's input): EAM::hessian
// (eam.cpp:122-233), Hessian::mass_weight (hessian.hpp:136-143) and Hessian::eigenvalues
// (hessian.hpp:86-93; the reference calls Eigen's SelfAdjointEigenSolver), as used by Master for
// Mechanism::kinetic_pre (find.cpp:838-871) and the minimum's log-product (find.cpp:1094-1144).
//
// Assembly: the analytic block, row by row.  With u = (r_a - r_g) / r along a listed pair,
//   H = sum over pairs of K (+K on the diagonal blocks, -K between the two atoms),
//       K = k'' u u^T + (m / r) (I - u u^T),  m = V' + F'_g phi'_{a->g} + F'_a phi'_{g->a}, k'' the same of second derivatives,
//     + sum over atoms b, frozen ones included, of F''_b (grad rho_b)(grad rho_b)^T.
// D holds dF'_b by moved coordinate for every atom b next to a mobile one; a row of H is then the pair
// blocks plus a short sum of rows of D (one per neighbour), so both kernels stream whole rows.  Mobile atoms scattered
// through a large system have up to 66 times as many neighbours: D is made for a panel of columns at a time, of at
// most HESS_PANEL, instead of 20 times H.  Assembly from
// the columns' Hessian-vector products took five launches and two passes over the whole system for
// each of the 3M coordinates: 11 ms at 120 mobile atoms in a 2000-atom cell, now 60 us.
//
// Eigenvalues: Householder reduction to tridiagonal form (Golub & Van Loan, Matrix Computations, Alg. 8.3.1),
// one launch a column that applies the previous reflection and multiplies by the next one in the same
// pass over the block; then each eigenvalue by multisection on Sturm counts (Givens' bisection), a
// wavefront per eigenvalue testing 64 points of its interval at once.  Both are
// backward stable: errors of a few units of 1e-16 of the largest eigenvalue.  Bound by one launch per column, 5 us, up
// to some 550 coordinates; above, a column also waits for the shrinking block and its vectors from the caches (8 us
// at 780 coordinates, 11 at 1200).  Cyclic Jacobi rotations
// needed ten sweeps of 3M rounds of two launches: 36 ms at 360 coordinates.
#include <algorithm>
#include <cmath>
#include <vector>

#include "vecops.hpp"

namespace flyg {

  namespace {

    constexpr int NTB = 256;
    constexpr std::size_t HESS_KEEP = 64u << 20;   // largest workspace kept in the potential handle between calls
    constexpr std::size_t HESS_PANEL = 256u << 20;   // largest panel of D

    constexpr int EC = 256;   // neighbour entries staged at a time

    // F' and F'' of every atom.
    template <int L>
    __global__ __launch_bounds__(NTB) void k_embed(EAMTables T, Shifts S, PairArgs A, double2* __restrict__ ff,
                                                   unsigned* __restrict__ err) {
      long const gid = blockIdx.x * static_cast<long>(NTB) + threadIdx.x;
      long const i = gid / L;
      int const lane = static_cast<int>(gid % L);
      bool const act = i < A.n;
      unsigned e = 0;
      double rho = 0;
      int ti = 0;
      if (act) {
        double4 const pi = A.pos[i];
        ti = A.t0 < 0 ? checked_type(A.types[i], T.ntypes, e) : A.t0;
        int const c = min(A.cnt[i], A.K);
        for (int k = lane; k < c; k += L) {
          unsigned const en = A.nbr[i * static_cast<long>(A.K) + k];
          unsigned const j = en & NB_IDX_MASK;
          double3 const sh = S.of(en >> NB_SHIFT_BITS);
          double4 const pj = A.pos[j];
          double const dx = (pj.x + sh.x) - pi.x, dy = (pj.y + sh.y) - pi.y, dz = (pj.z + sh.z) - pi.z;
          double const r2 = dx * dx + dy * dy + dz * dz;
          if (r2 < T.rc2) {
            int const tj = A.t0 < 0 ? checked_type(A.types[j], T.ntypes, e) : A.t0;
            rho += spl64<0>(T, T.phi[tj + T.ntypes * ti], sqrt(r2), e);
          }
        }
      }
      rho = group_sum<L>(rho);
      if (act && lane == 0) ff[i] = make_double2(spl64<1>(T, T.F[ti], rho, e), spl64<2>(T, T.F[ti], rho, e));
      if (e) atomicOr(err, e);
    }

    // Marks the mobile atoms and their neighbours (one wavefront per mobile atom).
    __global__ void k_mark(PairArgs A, int const* __restrict__ atoms, long nm, int* __restrict__ mark) {
      long const w = (blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x) / 64;
      int const lane = threadIdx.x & 63;
      if (w >= nm) return;
      long const i = atoms[w];
      if (lane == 0) mark[i] = 1;
      int const c = min(A.cnt[i], A.K);
      for (int k = lane; k < c; k += 64) mark[A.nbr[i * static_cast<long>(A.K) + k] & NB_IDX_MASK] = 1;
    }

    // loc = exclusive scan of the marks: the atom of each row of D.
    __global__ void k_region(int const* __restrict__ loc, long n, int* __restrict__ region) {
      long const i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
      if (i < n && loc[i + 1] > loc[i]) region[loc[i]] = static_cast<int>(i);
    }

    struct Pair {
      double ux, uy, uz, r;
      int j, ti, tj;
      bool in;
    };

    __device__ inline Pair pair_at(EAMTables const& T, Shifts const& S, PairArgs const& A, long i, double4 const& pi, int ti,
                                   int k, unsigned& e) {
      Pair p;
      unsigned const en = A.nbr[i * static_cast<long>(A.K) + k];
      p.j = static_cast<int>(en & NB_IDX_MASK);
      double3 const sh = S.of(en >> NB_SHIFT_BITS);
      double4 const pj = A.pos[p.j];
      double const dx = (pj.x + sh.x) - pi.x, dy = (pj.y + sh.y) - pi.y, dz = (pj.z + sh.z) - pi.z;
      double const r2 = dx * dx + dy * dy + dz * dz;
      p.in = r2 < T.rc2;
      p.r = p.in ? sqrt(r2) : 1.0;
      p.ux = dx / p.r;
      p.uy = dy / p.r;
      p.uz = dz / p.r;
      p.ti = ti;
      p.tj = A.t0 < 0 ? checked_type(A.types[p.j], T.ntypes, e) : A.t0;
      return p;
    }

    // Row b of D: F''_b d rho_b / d (coordinate) for mobile coordinates c0 .. c0 + w - 1.  One workgroup per region atom:
    // its entries are staged in LDS, then every thread sums those that touch its columns, in row order.
    __global__ __launch_bounds__(NTB) void k_drow(EAMTables T, Shifts S, PairArgs A, double2 const* __restrict__ ff,
                                                  int const* __restrict__ region, int const* __restrict__ mob, long c0,
                                                  long w, double* __restrict__ D, unsigned* __restrict__ err) {
      __shared__ double s_g[3][EC];
      __shared__ int s_m[EC];
      long const b = region[blockIdx.x];
      unsigned e = 0;
      double4 const pb = A.pos[b];
      int const tb = A.t0 < 0 ? checked_type(A.types[b], T.ntypes, e) : A.t0;
      int const mb = mob[b];
      double const fpp = ff[b].y;
      int const c = min(A.cnt[b], A.K);
      double* row = D + blockIdx.x * w;
      for (int k0 = 0; k0 == 0 || k0 < c; k0 += EC) {
        int const nk = min(EC, c - k0);
        __syncthreads();
        for (int k = threadIdx.x; k < nk; k += NTB) {
          Pair const p = pair_at(T, S, A, b, pb, tb, k0 + k, e);
          double const f = p.in ? fpp * spl64<1>(T, T.phi[p.tj + T.ntypes * tb], p.r, e) : 0.0;
          s_g[0][k] = f * p.ux;
          s_g[1][k] = f * p.uy;
          s_g[2][k] = f * p.uz;
          s_m[k] = p.in ? mob[p.j] : -2;
        }
        __syncthreads();
        for (long q = threadIdx.x; q < w; q += NTB) {
          int const m = static_cast<int>((c0 + q) / 3), d = static_cast<int>((c0 + q) % 3);
          double v = k0 ? row[q] : 0.0;
          if (m == mb) {
            for (int k = 0; k < nk; ++k) v += (s_m[k] == m ? s_g[d][k] : 0.0) - s_g[d][k];
          } else {
            for (int k = 0; k < nk; ++k)
              if (s_m[k] == m) v += s_g[d][k];
          }
          row[q] = v;
        }
      }
      if (e) atomicOr(err, e);
    }

    // Columns c0 .. c0 + w - 1 of rows 3g .. 3g + 2 of the mass-weighted block.  One workgroup per mobile atom g.
    __global__ __launch_bounds__(NTB) void k_hrow(EAMTables T, Shifts S, PairArgs A, double2 const* __restrict__ ff,
                                                  int const* __restrict__ atoms, int const* __restrict__ mob,
                                                  int const* __restrict__ loc, double const* __restrict__ rmass, long n3m,
                                                  long c0, long w, double const* __restrict__ D, double* __restrict__ H,
                                                  unsigned* __restrict__ err) {
      __shared__ double s_u[3][EC], s_g[EC], s_a[EC], s_k[EC], s_t[EC];   // u, phi'_{a->g}, phi'_{g->a}, k'' - m / r, m / r
      __shared__ int s_m[EC], s_l[EC];
      int const mg = static_cast<int>(blockIdx.x);
      long const g = atoms[mg];
      unsigned e = 0;
      double4 const pg = A.pos[g];
      int const tg = A.t0 < 0 ? checked_type(A.types[g], T.ntypes, e) : A.t0;
      double const fg = ff[g].x;
      int const c = min(A.cnt[g], A.K);
      double const* Dg = D + static_cast<long>(loc[g]) * w;
      double* h0 = H + 3l * mg * n3m;
      for (int k0 = 0; k0 == 0 || k0 < c; k0 += EC) {
        int const nk = min(EC, c - k0);
        __syncthreads();
        for (int k = threadIdx.x; k < nk; k += NTB) {
          Pair const p = pair_at(T, S, A, g, pg, tg, k0 + k, e);
          double ga = 0, gb = 0, kk = 0, tt = 0;
          if (p.in) {
            SplineDesc const& sv = T.V[vidx(T, tg, p.tj)];
            SplineDesc const& sa = T.phi[p.tj + T.ntypes * tg];
            SplineDesc const& sb = T.phi[tg + T.ntypes * p.tj];
            double const fa = ff[p.j].x;
            ga = spl64<1>(T, sa, p.r, e);
            gb = spl64<1>(T, sb, p.r, e);
            double const m = spl64<1>(T, sv, p.r, e) + fg * ga + fa * gb;
            tt = m / p.r;
            kk = spl64<2>(T, sv, p.r, e) + fg * spl64<2>(T, sa, p.r, e) + fa * spl64<2>(T, sb, p.r, e) - tt;
          }
          s_u[0][k] = p.ux;
          s_u[1][k] = p.uy;
          s_u[2][k] = p.uz;
          s_g[k] = ga;
          s_a[k] = gb;
          s_k[k] = kk;
          s_t[k] = tt;
          s_m[k] = p.in ? mob[p.j] : -2;
          s_l[k] = p.in ? loc[p.j] : loc[g];
        }
        __syncthreads();
        for (long at = threadIdx.x; at < w; at += NTB) {
          long const col = c0 + at;
          int const m = static_cast<int>(col / 3), d = static_cast<int>(col % 3);
          double const dg = Dg[at], rc = rmass[col];
          double h[3] = {0, 0, 0};
#pragma unroll 4
          for (int k = 0; k < nk; ++k) {
            double const q = s_g[k] * dg + s_a[k] * D[s_l[k] * w + at];
#pragma unroll
            for (int r = 0; r < 3; ++r) h[r] -= s_u[r][k] * q;
            double const on = (m == mg ? 1.0 : 0.0) - (m == s_m[k] ? 1.0 : 0.0);
            if (on != 0.0) {
              double const ud = s_u[d][k] * s_k[k];
#pragma unroll
              for (int r = 0; r < 3; ++r) h[r] += on * (s_u[r][k] * ud + (r == d ? s_t[k] : 0.0));
            }
          }
#pragma unroll
          for (int r = 0; r < 3; ++r) {
            double const v = h[r] * (rmass[3 * mg + r] * rc);
            h0[r * n3m + col] = k0 ? h0[r * n3m + col] + v : v;
          }
        }
      }
      if (e) atomicOr(err, e);
    }

    // Keep the lower triangle: H[c][r] = H[r][c] for r > c.
    __global__ void k_mirror_lower(double* __restrict__ H, long n) {
      long idx = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
      if (idx >= n * n) return;
      long r = idx / n, c = idx % n;
      if (r > c) H[c * n + r] = H[r * n + c];
    }

    // Block sums of two values, to every thread.
    __device__ inline void sum2(double& x, double& y, double (*sh)[NTB / 64]) {
      x = group_sum<64>(x);
      y = group_sum<64>(y);
      __syncthreads();
      if ((threadIdx.x & 63) == 0) {
        sh[0][threadIdx.x >> 6] = x;
        sh[1][threadIdx.x >> 6] = y;
      }
      __syncthreads();
      x = y = 0;
#pragma unroll
      for (int w = 0; w < NTB / 64; ++w) {
        x += sh[0][w];
        y += sh[1][w];
      }
    }

    // Step k of the reduction.  A holds the block before reflection k - 1 is applied (its vector v, scale b and
    // product p = A v are in vp, bt and pp); rows above k are done.  Every workgroup for itself: w = b p - (b^2 (p.v) / 2) v,
    // row k of the updated block, its diagonal and the next reflection; then, a wavefront per row,
    // A_ij -= v_i w_j + w_i v_j and the row's part of A v_new.  Row k itself is only read.
    //
    // A step is a launch and a chain of loads, two block sums and a row sum: what it costs at 360
    // coordinates is latency.  NC > 0 (blocks of up to 64 NC coordinates): vectors and rows are loaded at once
    // before the first sum, v, w and the new vector wait in LDS (6.4 -> 4.6 us a step).  NC = 0: any size,
    // everything read again from the caches where it is used.
    template <int NC>
    __global__ __launch_bounds__(NTB) void k_tridiag(double* __restrict__ A, long n, long k, double const* __restrict__ vp,
                                                     double const* __restrict__ pp, double const* __restrict__ bt,
                                                     double* __restrict__ vn, double* __restrict__ pn,
                                                     double* __restrict__ bn, double* __restrict__ diag,
                                                     double* __restrict__ off) {
      constexpr int NV = NC > 0 ? (64 * NC + NTB - 1) / NTB : 1;   // elements of a vector per thread
      __shared__ double sh[2][2][NTB / 64];
      __shared__ double sv[NC > 0 ? 64 * NC : 1], sw[NC > 0 ? 64 * NC : 1], sx[NC > 0 ? 64 * NC : 1];
      double const* Ak = A + k * n;
      bool const first = k == 0;
      double const b = first ? 0.0 : *bt;
      int const lane = threadIdx.x & 63;
      long const waves = static_cast<long>(gridDim.x) * (NTB / 64);
      long const i0 = k + 1 + blockIdx.x * (NTB / 64) + (threadIdx.x >> 6);   // this wavefront's first row
      double ev[NV], ep[NV], ea[NV];   // v, p and row k
      double row[NC > 0 ? NC : 1];
      if constexpr (NC > 0) {
#pragma unroll
        for (int u = 0; u < NV; ++u) {
          long const j = k + threadIdx.x + u * NTB;
          bool const in = j < n;
          ev[u] = in && !first ? vp[j] : 0.0;
          ep[u] = in && !first ? pp[j] : 0.0;
          ea[u] = in ? Ak[j] : 0.0;
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          long const j = k + 1 + lane + 64 * c;
          row[c] = i0 < n && j < n ? A[i0 * n + j] : 0.0;
        }
      }
      double pv = 0, dummy = 0;
      if constexpr (NC > 0) {
#pragma unroll
        for (int u = 0; u < NV; ++u) pv += ep[u] * ev[u];
      } else {
        if (!first)
          for (long j = k + threadIdx.x; j < n; j += NTB) pv += pp[j] * vp[j];
      }
      sum2(pv, dummy, sh[0]);
      double const kk = 0.5 * b * b * pv;
      if constexpr (NC > 0) {
#pragma unroll
        for (int u = 0; u < NV; ++u) {
          int const q = threadIdx.x + u * NTB;   // place of element k + q
          if (q < 64 * NC) {
            sv[q] = ev[u];
            sw[q] = b * ep[u] - kk * ev[u];
          }
        }
        __syncthreads();
      }
      // v_j and w_j of the reflection before (zero at the first step).
      auto vw = [&](long j, double& v, double& w) {
        if constexpr (NC > 0) {
          v = sv[j - k];
          w = sw[j - k];
        } else {
          v = first ? 0.0 : vp[j];
          w = first ? 0.0 : b * pp[j] - kk * v;
        }
      };
      double vk, wk;
      vw(k, vk, wk);
      double ss = 0;
      if constexpr (NC > 0) {
#pragma unroll
        for (int u = 0; u < NV; ++u) {
          int const q = threadIdx.x + u * NTB;
          if (q < 64 * NC) {
            double const x = ea[u] - (vk * sw[q] + wk * sv[q]);   // row k of the updated block
            sx[q] = x;
            if (q >= 2) ss += x * x;
          }
        }
      }
      auto rowk = [&](long j, double& v, double& w) {
        vw(j, v, w);
        return Ak[j] - (vk * w + wk * v);
      };
      if constexpr (NC == 0)
        for (long j = k + 2 + threadIdx.x; j < n; j += NTB) {
          double v, w;
          double const x = rowk(j, v, w);
          ss += x * x;
        }
      double zero = 0;
      sum2(ss, zero, sh[1]);
      double x0, x1;
      if constexpr (NC > 0) {
        x0 = sx[0];
        x1 = sx[1];
      } else {
        double v, w;
        x0 = rowk(k, v, w);
        x1 = rowk(k + 1, v, w);
      }
      double alpha = x1, top = 0, beta = 0;
      if (ss != 0.0) {
        alpha = -copysign(sqrt(ss + x1 * x1), x1);
        top = x1 - alpha;
        beta = 2.0 / (ss + top * top);
      }
      auto next = [&](long j) {   // new reflection's vector (zero where there is none)
        double x;
        if constexpr (NC > 0) {
          x = sx[j - k];
        } else {
          double v, w;
          x = rowk(j, v, w);
        }
        return j == k + 1 ? top : (beta != 0.0 ? x : 0.0);
      };
      if (blockIdx.x == 0) {
        if (threadIdx.x == 0) {
          diag[k] = x0;
          off[k] = alpha;
          *bn = beta;
        }
        for (long j = k + 1 + threadIdx.x; j < n; j += NTB) vn[j] = next(j);
      }
      for (long i = i0; i < n; i += waves) {
        double vi, wi;
        vw(i, vi, wi);
        double* Ai = A + i * n;
        double p = 0;
        auto one = [&](long j, double a0) {
          double v, w;
          vw(j, v, w);
          double const a = a0 - (vi * w + wi * v);
          Ai[j] = a;
          p += a * next(j);
        };
        if constexpr (NC > 0) {
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            long const j = k + 1 + lane + 64 * c;
            if (j < n) one(j, i == i0 ? row[c] : Ai[j]);
          }
        } else {
          for (long j = k + 1 + lane; j < n; j += 64) one(j, Ai[j]);
        }
        p = group_sum<64>(p);
        if (lane == 0) pn[i] = p;
      }
    }

    // The last 2 x 2 (or 1 x 1) block once no reflection is left.
    __global__ void k_tridiag_end(double const* __restrict__ A, long n, double const* __restrict__ vp,
                                  double const* __restrict__ pp, double const* __restrict__ bt, double* __restrict__ diag,
                                  double* __restrict__ off) {
      if (threadIdx.x) return;
      long const k = n >= 2 ? n - 2 : 0;
      bool const none = n < 3;
      double const b = none ? 0.0 : *bt;
      double pv = 0;
      if (!none)
        for (long j = k; j < n; ++j) pv += pp[j] * vp[j];
      double const kk = 0.5 * b * b * pv;
      for (long i = k; i < n; ++i) {
        double const vi = none ? 0.0 : vp[i], wi = none ? 0.0 : b * pp[i] - kk * vi;
        diag[i] = A[i * n + i] - 2.0 * (vi * wi);
        if (i > k) {
          double const v = none ? 0.0 : vp[k], w = none ? 0.0 : b * pp[k] - kk * v;
          off[k] = A[k * n + i] - (vi * w + wi * v);
        }
      }
    }

    // Gershgorin bounds of the tridiagonal matrix and, for the Sturm counts, the matrix scaled by a power of two to a
    // norm in [1/2, 1) (exact): ds, and e2 = squares of the off-diagonal (one workgroup).  lim = (low, high,
    // scale) in scaled units.
    __global__ __launch_bounds__(NTB) void k_bounds(double const* __restrict__ d, double const* __restrict__ off, long n,
                                                    double* __restrict__ ds, double* __restrict__ e2,
                                                    double* __restrict__ lim) {
      __shared__ double s0[NTB / 64], s1[NTB / 64];
      __shared__ int s2[NTB / 64];
      double lo = INFINITY, hi = -INFINITY;
      int bad = 0;
      for (long i = threadIdx.x; i < n; i += NTB) {
        double const l = i > 0 ? fabs(off[i - 1]) : 0.0, r = i + 1 < n ? fabs(off[i]) : 0.0;
        double const a = d[i] - (l + r), z = d[i] + (l + r);
        bad |= !isfinite(a) || !isfinite(z);
        lo = fmin(lo, a);
        hi = fmax(hi, z);
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        lo = fmin(lo, __shfl_xor(lo, o, 64));
        hi = fmax(hi, __shfl_xor(hi, o, 64));
        bad |= __shfl_xor(bad, o, 64);
      }
      if ((threadIdx.x & 63) == 0) {
        s0[threadIdx.x >> 6] = lo;
        s1[threadIdx.x >> 6] = hi;
        s2[threadIdx.x >> 6] = bad;
      }
      __syncthreads();
      for (int q = 0; q < NTB / 64; ++q) {
        lo = fmin(lo, s0[q]);
        hi = fmax(hi, s1[q]);
        bad |= s2[q];
      }
      int ex = 0;
      double const norm = fmax(fabs(lo), fabs(hi));
      if (norm > 0) (void)frexp(norm, &ex);
      double const sc = ldexp(1.0, -ex), pad = 1e-15 * norm * sc + 1e-300;
      for (long i = threadIdx.x; i < n; i += NTB) {
        double const l = i > 0 ? off[i - 1] * sc : 0.0;
        ds[i] = d[i] * sc;
        e2[i] = fmax(l * l, 1e-36);   // couples i - 1 and i; a coupling of 1e-18 of the norm keeps p from sticking at zero
      }
      if (threadIdx.x == 0) {
        lim[0] = bad ? NAN : lo * sc - pad;
        lim[1] = bad ? NAN : hi * sc + pad;
        lim[2] = ldexp(1.0, ex);
      }
    }

    // Eigenvalue m of the tridiagonal matrix: one wavefront narrows its interval 65-fold per pass.  The number of
    // eigenvalues below x is the number of sign changes in p_i = (d_i - x) p_{i-1} - e_i^2 p_{i-2}: a chain of one
    // FMA a term (with q_i = p_i / p_{i-1} it is a division, 250 cycles).  The pair is rescaled every eight
    // terms, which cannot leave the range of a double for a matrix of norm 1; the sign of a term that vanishes does
    // not matter, since its neighbours' differ.  LDS: the matrix waits there (up to STURM_LDS coordinates), the
    // next eight terms are read while these are worked on.
    constexpr int STURM_PASSES = 9;   // 65^9 = 2^54: down to the rounding of the interval's own width
    constexpr int STURM_LDS = 3072;

    template <bool LDS>
    __global__ __launch_bounds__(NTB) void k_sturm(double const* __restrict__ d, double const* __restrict__ e2, long n,
                                                   double const* __restrict__ lim, double* __restrict__ out) {
      extern __shared__ double2 s_t[];   // (d, e2), padded by two groups with terms that keep p's sign
      if constexpr (LDS) {
        for (long i = threadIdx.x; i < n + 16; i += NTB) s_t[i] = i < n ? make_double2(d[i], e2[i]) : make_double2(2.0, 0.0);
        __syncthreads();
      }
      long const m = blockIdx.x * static_cast<long>(NTB / 64) +
                     __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
      int const lane = threadIdx.x & 63;
      if (m >= n) return;
      auto term = [&](long i) {
        if constexpr (LDS) return s_t[i];
        return i < n ? make_double2(d[i], e2[i]) : make_double2(2.0, 0.0);
      };
      double lo = lim[0], hi = lim[1];
      for (int pass = 0; pass < STURM_PASSES; ++pass) {
        double const x = lo + (hi - lo) * (static_cast<double>(lane + 1) / 65.0);
        double p0 = 0.0, p1 = 1.0;   // p_{i-2}, p_{i-1}
        int below = 0;
        double2 t8[8], n8[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) t8[u] = term(u);
        for (long i8 = 0; i8 < n; i8 += 8) {
#pragma unroll
          for (int u = 0; u < 8; ++u) n8[u] = term(i8 + 8 + u);
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            double const p = fma(t8[u].x - x, p1, -(t8[u].y * p0));
            below += static_cast<int>(static_cast<unsigned>(__double2hiint(p) ^ __double2hiint(p1)) >> 31);
            p0 = p1;
            p1 = p;
          }
          int const ex = max(__builtin_amdgcn_frexp_exp(p0), __builtin_amdgcn_frexp_exp(p1));
          p0 = ldexp(p0, -ex);
          p1 = ldexp(p1, -ex);
#pragma unroll
          for (int u = 0; u < 8; ++u) t8[u] = n8[u];
        }
        int const t = __popcll(__ballot(below <= m));   // points that eigenvalue m is not below
        double const nlo = __shfl(x, t > 0 ? t - 1 : 0, 64), nhi = __shfl(x, t < 64 ? t : 63, 64);
        if (t > 0) lo = nlo;
        if (t < 64) hi = nhi;
      }
      if (lane == 0) out[m] = 0.5 * (lo + hi) * lim[2];
    }

    unsigned blocks(long n, int t) { return static_cast<unsigned>((n + t - 1) / t); }

  }  // namespace

  // Returns the sorted eigenvalues of the mass-weighted Hessian block of the non-frozen atoms.
  std::vector<double> hessian_eigenvalues(flyg_eam_s& E, flyg_list_s& nl, uint32_t const* d_types,
                                          uint8_t const* d_frozen, std::vector<uint8_t> const& h_frozen,
                                          std::vector<uint32_t> const& h_types) {
    flyg_ctx_s& ctx = *E.ctx;
    hipStream_t st = ctx.stream;
    long const n = nl.n;
    std::vector<long> dof;
    std::vector<double> rmass;
    for (long a = 0; a < n; ++a) {
      if (h_frozen[a]) continue;
      uint32_t t = h_types[a];
      require(t < static_cast<uint32_t>(E.data.ntypes), "TypeID out of range");
      double m = E.data.mass[t];
      require(m > 0, "the potential gives a species no positive mass");
      for (int k = 0; k < 3; ++k) {
        dof.push_back(3 * a + k);
        rmass.push_back(1.0 / std::sqrt(m));
      }
    }
    long const n3m = static_cast<long>(dof.size());
    if (n3m == 0) return {};
    require(n3m <= 16384, "the Hessian block is limited to 16384 degrees of freedom");
    require(nl.built, "List used before rebuild");
    require(E.tab.rc <= nl.rc, "r_cut is bigger than the internal r_cut of the list");
    long const nm = n3m / 3;
    PairArgs const A = pair_args(E, nl, d_types, d_frozen);
    Shifts const S = shifts_of(nl.box);
    unsigned* err = ctx.dflags.get();

    // Mobile atoms, their neighbours (the rows of D) and F', F''.
    std::vector<int> host(static_cast<std::size_t>(n + nm), -1);   // mobile index by atom, then the mobile atoms
    for (long q = 0; q < nm; ++q) {
      long const a = dof[3 * q] / 3;
      host[a] = static_cast<int>(q);
      host[n + q] = static_cast<int>(a);
    }
    long const nloc = scan_room(n + 1);
    E.hess_ids.reserve(2 * n + nloc + nm);
    int* loc = E.hess_ids.get();    // n + 1: marks, then their exclusive scan
    int* region = loc + nloc;       // up to n
    int* mob = region + n;
    int* atoms = mob + n;
    HIPCHK(hipMemcpyAsync(mob, host.data(), host.size() * sizeof(int), hipMemcpyHostToDevice, st));
    HIPCHK(hipMemsetAsync(loc, 0, (n + 1) * sizeof(int), st));
    k_mark<<<blocks(nm * 64, NTB), NTB, 0, st>>>(A, atoms, nm, loc);
    exclusive_scan(ctx, loc, loc, static_cast<int>(n + 1), nl.scan_tmp);
    k_region<<<blocks(n, NTB), NTB, 0, st>>>(loc, n, region);
    HIPCHK(hipMemcpyAsync(ctx.hflags + 2, loc + n, sizeof(int), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    long const nreg = static_cast<long>(ctx.hflags[2]);

    // One workspace: H, a panel of D, (F', F'') by atom, 1 / sqrt(m), and eight vectors of the reduction.
    long const panel = std::min(n3m, std::max<long>(1, HESS_PANEL / sizeof(double) / nreg));
    std::size_t const need = static_cast<std::size_t>(n3m) * (n3m + 9) + static_cast<std::size_t>(panel) * nreg + 2 * n + 16;
    DBuf<double> own;
    bool const keep = need * sizeof(double) <= HESS_KEEP;
    DBuf<double>& work = keep ? E.hess : own;
    work.reserve(need);
    double2* ff = reinterpret_cast<double2*>(work.get());
    double* H = work.get() + 2 * n;
    double* D = H + n3m * n3m;
    double* rm = D + nreg * panel;
    double* v[2] = {rm + n3m, rm + 2 * n3m};
    double* p[2] = {rm + 3 * n3m, rm + 4 * n3m};
    double* diag = rm + 5 * n3m;
    double* off = rm + 6 * n3m;
    double* e2 = rm + 7 * n3m;
    double* lam = rm + 8 * n3m;
    double* bt[2] = {rm + 9 * n3m, rm + 9 * n3m + 1};
    double* lim = rm + 9 * n3m + 2;
    HIPCHK(hipMemcpyAsync(rm, rmass.data(), n3m * sizeof(double), hipMemcpyHostToDevice, st));
    k_embed<8><<<blocks(n * 8, NTB), NTB, 0, st>>>(E.tab, S, A, ff, err);
    for (long c0 = 0; c0 < n3m; c0 += panel) {
      long const w = std::min(panel, n3m - c0);
      k_drow<<<static_cast<unsigned>(nreg), NTB, 0, st>>>(E.tab, S, A, ff, region, mob, c0, w, D, err);
      k_hrow<<<static_cast<unsigned>(nm), NTB, 0, st>>>(E.tab, S, A, ff, atoms, mob, loc, rm, n3m, c0, w, D, H, err);
    }
    k_mirror_lower<<<blocks(n3m * n3m, NTB), NTB, 0, st>>>(H, n3m);
    for (long k = 0; k + 2 < n3m; ++k) {
      long const rows = n3m - k - 1;
      unsigned const g = static_cast<unsigned>(std::min<long>((rows + NTB / 64 - 1) / (NTB / 64), 512));
      auto step = [&](auto f) {
        f<<<g, NTB, 0, st>>>(H, n3m, k, v[k & 1], p[k & 1], bt[k & 1], v[(k + 1) & 1], p[(k + 1) & 1], bt[(k + 1) & 1], diag,
                             off);
      };
      long const left = n3m - k;   // coordinates of the block, row k among them
      left <= 128 ? step(k_tridiag<2>) : left <= 256 ? step(k_tridiag<4>) : left <= 512 ? step(k_tridiag<8>)
                                       : step(k_tridiag<0>);
    }
    k_tridiag_end<<<1, 64, 0, st>>>(H, n3m, v[n3m & 1], p[n3m & 1], bt[n3m & 1], diag, off);
    k_bounds<<<1, NTB, 0, st>>>(diag, off, n3m, rm, e2, lim);   // rm: the scaled diagonal (the masses are done with)
    if (n3m <= STURM_LDS) {
      k_sturm<true><<<blocks(n3m, NTB / 64), NTB, (n3m + 16) * sizeof(double2), st>>>(rm, e2, n3m, lim, lam);
    } else {
      k_sturm<false><<<blocks(n3m, NTB / 64), NTB, 0, st>>>(rm, e2, n3m, lim, lam);
    }
    HIPCHK(hipGetLastError());
    std::vector<double> w(n3m);
    HIPCHK(hipMemcpyAsync(w.data(), lam, n3m * sizeof(double), hipMemcpyDeviceToHost, st));
    throw_flags(ctx.take_flags());   // synchronises
    std::sort(w.begin(), w.end());
    return w;
  }

}  // namespace flyg
