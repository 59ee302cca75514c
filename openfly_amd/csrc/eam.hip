// EAM / Finnis-Sinclair energy, gradient and Hessian-vector product on gfx950
// (replaces potential::EAM::energy / gradient / hessian, eam.cpp:33-233).
//
// Work mapping: systems with enough cells run in tiles (a workgroup stages a box of cells and its halo in LDS
// and walks 16-bit rows, see TILED PASSES below); smaller ones and calls that ask for it run row by row: L lanes
// (16 by default) of a wavefront cooperate on one atom's neighbour row (ELL layout, 32-bit packed entries), each
// lane striding the row by L.  Either way a row's sums go through Acc16's 16 slots, so the two give the same bits
// and results are reproducible run to run.  No atomics touch floating-point data.  In the rows positions are
// double4 (x, y, z, w): a neighbour gather is one 32-byte load, and pass 1 writes (x, y, z, F'(rho)) so pass 2 gets
// the neighbour's position and F' in that load (in the mixed form w holds F' as FP32 and the species, see
// pack_fp_type).
//
//   pass 1 (density):  rho_b = sum_a phi_{t_a->t_b}(r_ab);  F'_b = F_{t_b}'(rho_b)     (eam.cpp:62-86)
//   pass 2 (force):    dE/dr_g = -sum_a [V'(r) + F'_g phi'_{a->g}(r) + F'_a phi'_{g->a}(r)] (r_a - r_g)/r
//                      frozen atoms get exactly zero                                   (eam.cpp:90-120)
//   energy:            E = 1/2 sum_a sum_b V(r_ab) + sum_a F(rho_a), frozen included   (eam.cpp:33-51)
//   HVP (matrix-free directional derivative of the gradient along v, v masked to non-frozen atoms):
//      pass 1: drho_b = sum_a phi'_{a->b}(r) u.(v_a - v_b);  dF'_b = F''(rho_b) drho_b
//      pass 2: (Hv)_g = -sum_a [dm u + m (dv - u s)/r],  s = u.dv,  dv = v_a - v_g, u = (r_a - r_g)/r,
//              dm = (V'' + F'_g phi''_{a->g} + F'_a phi''_{g->a}) s + dF'_g phi'_{a->g} + dF'_a phi'_{g->a}
//      which is H v for the analytic Hessian of eam.cpp:122-233 (pinned against it in the tests).
#include <atomic>
#include <cstring>
#include <mutex>

#include "vecops.hpp"

namespace flyg {

  // t0 >= 0 selects the single-species kernels (constant table indices): always with one species
  // tabulated, and with several when the staged host types hold one species only.
  PairArgs pair_args(flyg_eam_s const& E, flyg_list_s& nl, uint32_t const* types, uint8_t const* frozen) {
    int t0 = E.tab.ntypes == 1 ? 0 : (types == E.types.get() ? E.staged_single : -1);
    return PairArgs{nl.pos.get(), nl.nbr.get(), nl.ncnt.get(), nl.K, nl.n, types, frozen, t0};
  }

  namespace {

    constexpr int NT = 256;

    // Mixed-form pass-1 output: the force pass uses F' only in FP32, so the w slot of (x, y, z, w) carries
    // F' as a float in its low 32 bits and the species in its high 32 bits, and a neighbour's species
    // arrives with its position (one gather less per pair).
    __device__ inline double pack_fp_type(float fp, int t) {
      return __longlong_as_double((static_cast<long long>(t) << 32) |
                                  static_cast<long long>(static_cast<unsigned>(__float_as_int(fp))));
    }
    __device__ inline float packed_fp(double w) {
      return __int_as_float(static_cast<int>(static_cast<unsigned>(__double_as_longlong(w) & 0xffffffffll)));
    }
    __device__ inline int packed_type(double w) { return static_cast<int>(__double_as_longlong(w) >> 32); }

    // One neighbour entry: image position difference and squared distance.
    struct PairGeo {
      double dx, dy, dz, r2, w;
      unsigned j;
    };

    __device__ inline PairGeo geo(Shifts const& S, double4 const* __restrict__ pos, unsigned en, double4 const& pi) {
      PairGeo p;
      p.j = en & NB_IDX_MASK;
      unsigned const code = en >> NB_SHIFT_BITS;
      double4 pj = pos[p.j];
      if (code != 13u) {   // image of a periodic neighbour (rows of interior atoms never take this branch)
        double3 sh = S.of(code);
        pj.x += sh.x;
        pj.y += sh.y;
        pj.z += sh.z;
      }
      p.dx = pj.x - pi.x;
      p.dy = pj.y - pi.y;
      p.dz = pj.z - pi.z;
      p.r2 = p.dx * p.dx + p.dy * p.dy + p.dz * p.dz;
      p.w = pj.w;
      return p;
    }

    // Walks lane `lane`'s share of a row (entries k = lane + m L): NS = 16 / L entries per step, entry m
    // of the step going to row-sum slot m (compile time), so every lane-count gives the same sums; for
    // L = 16 two entries per step share slot 0 in order.  All loads of a step are issued first.
    template <int L, typename F>
    __device__ inline void walk_row(unsigned const* __restrict__ row, int c, int lane, Shifts const& S,
                                    double4 const* __restrict__ pos, double4 const& pi, F&& one) {
      constexpr int NS = 16 / L;
      constexpr int U = NS == 1 ? 2 : NS;
      int m = 0;
      for (; lane + (m + U - 1) * L < c; m += U) {
        PairGeo p[U];
#pragma unroll
        for (int q = 0; q < U; ++q) p[q] = geo(S, pos, row[lane + (m + q) * L], pi);
#pragma unroll
        for (int q = 0; q < U; ++q) one(q % NS, p[q]);
      }
#pragma unroll
      for (int q = 0; q < U - 1; ++q)
        if (lane + (m + q) * L < c) one(q % NS, geo(S, pos, row[lane + (m + q) * L], pi));
    }

    // Density pass.  MIX (and not ENERGY): r and the density spline in FP32, sums in FP64.
    template <int L, bool MULTI, bool ENERGY, bool MIX>
    __global__ __launch_bounds__(NT) void k_density(EAMTables const* __restrict__ Tp, Shifts S, PairArgs A, double4* __restrict__ posf,
                                                    double* __restrict__ eatom, unsigned* __restrict__ err) {
      EAMTables const& T = *Tp;
      __shared__ SplineDesc s_phi[MAX_TYPES * MAX_TYPES], s_V[MAX_TYPES * MAX_TYPES];
      if (MULTI) {   // per-lane species pairs: table descriptors from LDS, not from the argument block
        int t = threadIdx.x;
        if (t < T.ntypes * T.ntypes) {
          s_phi[t] = T.phi[t];
          s_V[t] = T.V[t];
        }
        __syncthreads();
      }
      auto PHI = [&](int k) -> SplineDesc const& {
        if constexpr (MULTI) {
          return s_phi[k];
        } else {
          return T.phi[k];
        }
      };
      auto VV = [&](int k) -> SplineDesc const& {
        if constexpr (MULTI) {
          return s_V[k];
        } else {
          return T.V[k];
        }
      };
      long gid = xcd_block(blockIdx.x, gridDim.x) * static_cast<long>(NT) + threadIdx.x;
      long i = gid / L;
      int lane = static_cast<int>(gid % L);
      bool act = i < A.n;
      Acc16<L> rho, vs;
      unsigned e = 0;
      double4 pi = make_double4(0, 0, 0, 0);
      int ti = 0;
      if (act) {
        pi = A.pos[i];
        ti = MULTI ? checked_type(A.types[i], T.ntypes, e) : A.t0;
        int const c = min(A.cnt[i], A.K);
        unsigned const* row = A.nbr + i * static_cast<long>(A.K);
        walk_row<L>(row, c, lane, S, A.pos, pi, [&](int q, PairGeo const& p) {
          if (p.r2 < T.rc2) {
            int tj = MULTI ? checked_type(A.type_in_w ? static_cast<uint32_t>(p.w) : A.types[p.j], T.ntypes, e) : A.t0;
            if (MIX && !ENERGY) {
              float r2f = static_cast<float>(p.r2);
              float rf = r2f * __frsqrt_rn(r2f);
              rho.add_slot(q, static_cast<double>(spl32f<0>(T, PHI(tj + T.ntypes * ti), rf, e)));
            } else {
              double r = sqrt(p.r2);
              rho.add_slot(q, spl64<0>(T, PHI(tj + T.ntypes * ti), r, e));
              if (ENERGY) vs.add_slot(q, spl64<0>(T, VV(vidx(T, ti, tj)), r, e));
            }
          }
        });
      }
      double rt = rho.total();
      double vt = ENERGY ? vs.total() : 0.0;
      if (act && lane == 0) {
        double f, fp;
        spl64_ffp(T, T.F[ti], rt, f, fp, e);
        double const w = MIX && !ENERGY ? pack_fp_type(static_cast<float>(fp), ti) : fp;
        posf[i] = make_double4(pi.x, pi.y, pi.z, w);
        if (ENERGY) eatom[A.order ? A.order[i] : i] = 0.5 * vt + f;
      }
      if (e) atomicOr(err, e);
    }

    template <int L, bool MULTI, bool MIX>
    __global__ __launch_bounds__(NT) void k_force(EAMTables const* __restrict__ Tp, Shifts S, PairArgs A, double4 const* __restrict__ posf,
                                                  double* __restrict__ grad, unsigned* __restrict__ err) {
      EAMTables const& T = *Tp;
      __shared__ SplineDesc s_phi[MAX_TYPES * MAX_TYPES], s_V[MAX_TYPES * MAX_TYPES];
      if (MULTI) {   // per-lane species pairs: table descriptors from LDS, not from the argument block
        int t = threadIdx.x;
        if (t < T.ntypes * T.ntypes) {
          s_phi[t] = T.phi[t];
          s_V[t] = T.V[t];
        }
        __syncthreads();
      }
      auto PHI = [&](int k) -> SplineDesc const& {
        if constexpr (MULTI) {
          return s_phi[k];
        } else {
          return T.phi[k];
        }
      };
      auto VV = [&](int k) -> SplineDesc const& {
        if constexpr (MULTI) {
          return s_V[k];
        } else {
          return T.V[k];
        }
      };
      long gid = xcd_block(blockIdx.x, gridDim.x) * static_cast<long>(NT) + threadIdx.x;
      long i = gid / L;   // row: the atom, or its slot when A.order is set
      int lane = static_cast<int>(gid % L);
      bool inr = i < A.n;
      long const ia = inr && A.order ? A.order[i] : i;   // the atom, for its frozen flag and gradient
      unsigned e = 0;
      // The row's own data is loaded beside the frozen flag (not after it): the flag waits on `order`.
      double4 pi = make_double4(0.0, 0.0, 0.0, 0.0);
      int ti = MULTI ? 0 : A.t0;
      int c = 0;
      if (inr) {
        pi = posf[i];
        c = min(A.cnt[i], A.K);
        // Mixed form: the species the density pass packed beside F' (checked there).
        if (MULTI) ti = MIX ? packed_type(pi.w) : checked_type(A.types[i], T.ntypes, e);
      }
      bool act = inr && !A.frozen[ia];
      Acc16<L> gx, gy, gz;
      if (act) {
        unsigned const* row = A.nbr + i * static_cast<long>(A.K);
        walk_row<L>(row, c, lane, S, posf, pi, [&](int q, PairGeo const& p) {
          if (p.r2 < T.rc2) {
            int tj = MULTI ? (MIX ? packed_type(p.w) : checked_type(A.types[p.j], T.ntypes, e)) : A.t0;
            double cf;
            if (MIX) {
              float r2f = static_cast<float>(p.r2);
              float rinv = __frsqrt_rn(r2f);
              float rf = r2f * rinv;
              float vp = spl32f<1>(T, VV(vidx(T, ti, tj)), rf, e);
              float pa = spl32f<1>(T, PHI(tj + T.ntypes * ti), rf, e);
              // phi_{g->a} is phi_{a->g} for a same-species pair: no second table load.
              float pb = MULTI && ti != tj ? spl32f<1>(T, PHI(ti + T.ntypes * tj), rf, e) : pa;
              float mag = vp + packed_fp(pi.w) * pa + packed_fp(p.w) * pb;
              cf = static_cast<double>(mag * rinv);
            } else {
              double r = sqrt(p.r2);
              double vp = spl64<1>(T, VV(vidx(T, ti, tj)), r, e);
              double pa = spl64<1>(T, PHI(tj + T.ntypes * ti), r, e);
              double pb = MULTI && ti != tj ? spl64<1>(T, PHI(ti + T.ntypes * tj), r, e) : pa;
              cf = (vp + pi.w * pa + p.w * pb) / r;
            }
            gx.add_slot(q, -cf * p.dx);
            gy.add_slot(q, -cf * p.dy);
            gz.add_slot(q, -cf * p.dz);
          }
        });
      }
      double tx = gx.total(), ty = gy.total(), tz = gz.total();
      if (L >= 3 && inr && lane < 3) {
        double v = lane == 0 ? tx : (lane == 1 ? ty : tz);
        grad[3 * ia + lane] = act ? v : 0.0;
      }
      if (L < 3 && inr && lane == 0) {
        grad[3 * ia] = act ? tx : 0.0;
        grad[3 * ia + 1] = act ? ty : 0.0;
        grad[3 * ia + 2] = act ? tz : 0.0;
      }
      if (e) atomicOr(err, e);
    }

    // ---- Tiled passes -------------------------------------------------------------------------------
    // One workgroup per tile of cells (TileGrid).  It stages the entries of the tile's halo in LDS, image
    // shifts applied, and walks the rows of the tile's atoms 16 lanes a row through 16-bit indices into the stage.
    //
    // Why: the row-gather kernels above are bound by L1 lookups, one cache line a clock and CU.  64 pairs need 128 of
    // them for the neighbours' positions, 64 per spline segment read and 8 for the row; at 54.5k atoms the
    // density pass counts 8.8M lookups, 14 us of its 18.  From LDS a position costs no lookup, and a 2x2x2
    // tile stages eight entries per atom, read in order, where it gathered 65.  A stage of one cell (27 entries per
    // atom, little work between barriers) was slower than the gathers.
    // Entries, their order and every expression are those of the row-gather kernels: the same bits.

    constexpr int TT = 512;   // threads: 32 rows at a time

    struct TileArgs {
      TileGrid G;
      int const* cstart;       // entries by cell, then (from nc1) real slots by cell
      unsigned const* sslot;
      unsigned const* rows;
      int rowW;                // words a row
      int K;
      int const* cnt;          // by slot
      int const* order;
      double4 const* pos;      // by slot; w: species (several species, density pass) or F'
      uint32_t const* types;   // by slot (several species)
      uint8_t const* frozen;   // by atom
      int t0;
      int cap;                 // entries of room in the stage
    };

    struct TileLds {
      int ls[16], off[17];     // halo lines: first sorted entry, place in the stage
      int os[16], oo[17];      // own lines: first slot, rows before it
    };

    // The last of 16 lines that starts at or before x.
    __device__ inline int line_of(int const* off, int x) {
      int q = 0;
#pragma unroll
      for (int b = 8; b > 0; b >>= 1)
        if (off[q + b] <= x) q += b;
      return q;
    }

    // Fills the line tables and the stage (xy, zw; types where `st` is given).  Ends with a barrier.
    template <typename F>
    __device__ inline void stage_tile(TileArgs const& A, Shifts const& S, TileLds& L, double2* xy, double2* zw, F&& extra) {
      int const t = static_cast<int>(xcd_block(blockIdx.x, gridDim.x));
      if (threadIdx.x < 64) {   // lanes 0..15 the halo's lines, 16..31 the tile's own
        int const q = threadIdx.x & 15;
        bool const own = threadIdx.x >= 16;
        int cb, ce;
        A.G.line(!own, t % A.G.nt[0], t / A.G.nt[0] % A.G.nt[1], t / (A.G.nt[0] * A.G.nt[1]), q, cb, ce);
        int const* c = A.cstart + (own ? A.G.nc1 : 0);
        int const b = c[cb], len = c[ce] - b;
        int incl = len;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
          int const v = __shfl_up(incl, o, 16);
          if (q >= o) incl += v;
        }
        if (threadIdx.x < 16) {
          L.ls[q] = b;
          L.off[q] = incl - len;
          if (q == 15) L.off[16] = incl;
        } else if (threadIdx.x < 32) {
          L.os[q] = b - A.cstart[A.G.nc1];
          L.oo[q] = incl - len;
          if (q == 15) L.oo[16] = incl;
        }
      }
      __syncthreads();
      int const total = min(L.off[16], A.cap);
      for (int e0 = threadIdx.x; e0 < total; e0 += 4 * TT) {
        unsigned en[4];
        double4 p[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          int const e = e0 + u * TT;
          if (e < total) {
            int const q = line_of(L.off, e);
            en[u] = A.sslot[L.ls[q] + (e - L.off[q])];
          }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (e0 + u * TT < total) p[u] = A.pos[en[u] & NB_IDX_MASK];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          int const e = e0 + u * TT;
          if (e < total) {
            unsigned const code = en[u] >> NB_SHIFT_BITS;
            if (code != 13u) {
              double3 const sh = S.of(code);
              p[u].x += sh.x;
              p[u].y += sh.y;
              p[u].z += sh.z;
            }
            xy[e] = make_double2(p[u].x, p[u].y);
            zw[e] = make_double2(p[u].z, p[u].w);
            extra(e, en[u] & NB_IDX_MASK);
          }
        }
      }
      __syncthreads();
    }

    // NB entries of a lane's row: geometry, and whether each is a pair within the cut-off.
    template <int NB>
    struct Pairs {
      PairGeo p[NB];
      bool in[NB];
    };

    // Lane l of 16 walks entries l, l + 16, ... of a row.  Entries go to one() four at a time so that their table
    // loads are in flight together (entry by entry a row is a chain of five L2 round trips); those past the row's end
    // or the cut-off are marked, not branched around.  The number of steps is that of the wavefront's
    // longest row, so no control flow diverges.  Every lane of the wavefront must call it (lanes without a row with
    // c = 0).  The next group's words are loaded ahead.
    template <typename F>
    __device__ inline void walk_tile_grouped(unsigned const* __restrict__ row, int c, int l, double4 const& pi, double rc2,
                                             double2 const* xy, double2 const* zw, F&& one) {
      int const c0 = __builtin_amdgcn_readlane(c, 0), c1 = __builtin_amdgcn_readlane(c, 16);
      int const c2 = __builtin_amdgcn_readlane(c, 32), c3 = __builtin_amdgcn_readlane(c, 48);
      int const steps = (max(max(c0, c1), max(c2, c3)) + 15) / 16;
      unsigned w0 = 0, w1 = 0;
      if (c > 0) w0 = row[l];
      if (c > 32) w1 = row[16 + l];
      auto group = [&](auto nb, unsigned a, unsigned b, int k) {
        constexpr int NB = decltype(nb)::value;
        Pairs<NB> G;
#pragma unroll
        for (int n = 0; n < NB; ++n) {
          unsigned const word = n < 2 ? a : b;
          bool const valid = k + 16 * n < c;
          unsigned const j = valid ? ((n & 1) ? word >> 16 : word & 0xffffu) : 0u;
          PairGeo& p = G.p[n];
          double2 const u = xy[j], v = zw[j];
          p.dx = u.x - pi.x;
          p.dy = u.y - pi.y;
          p.dz = v.x - pi.z;
          p.w = v.y;
          p.j = j;
          p.r2 = p.dx * p.dx + p.dy * p.dy + p.dz * p.dz;
          G.in[n] = valid && p.r2 < rc2;
        }
        one(G);
      };
      for (int s = 0; s < steps; s += 4) {
        int const k = 16 * s + l, left = steps - s;
        unsigned n0 = 0, n1 = 0;
        if (16 * (s + 4) < c) n0 = row[8 * (s + 4) + l];
        if (16 * (s + 6) < c) n1 = row[8 * (s + 6) + l];
        if (left >= 4) {
          group(std::integral_constant<int, 4>{}, w0, w1, k);
        } else if (left == 1) {
          group(std::integral_constant<int, 1>{}, w0, 0u, k);
        } else {
          group(std::integral_constant<int, 2>{}, w0, 0u, k);
          if (left == 3) group(std::integral_constant<int, 1>{}, w1, 0u, k + 32);
        }
        w0 = n0;
        w1 = n1;
      }
    }

    // The same, entry by entry, pairs outside the cut-off branched around: for the forms whose table loads and
    // arithmetic of several entries would not fit in the registers that leave three workgroups a CU.
    template <typename F>
    __device__ inline void walk_tile(unsigned const* __restrict__ row, int c, int l, double4 const& pi, double rc2,
                                     double2 const* xy, double2 const* zw, F&& one) {
      unsigned w[4];   // the first 128 entries: a row's words are in flight together
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = 32 * u < c ? row[16 * u + l] : 0u;
      auto pair = [&](unsigned word, int k) {
        unsigned const j[2] = {word & 0xffffu, word >> 16};
        PairGeo p[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
          if (k + 16 * h < c) {
            double2 const a = xy[j[h]], b = zw[j[h]];
            p[h].dx = a.x - pi.x;
            p[h].dy = a.y - pi.y;
            p[h].dz = b.x - pi.z;
            p[h].w = b.y;
            p[h].j = j[h];
          }
#pragma unroll
        for (int h = 0; h < 2; ++h)
          if (k + 16 * h < c) {
            p[h].r2 = p[h].dx * p[h].dx + p[h].dy * p[h].dy + p[h].dz * p[h].dz;
            if (p[h].r2 < rc2) one(p[h]);
          }
      };
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (32 * u < c) pair(w[u], 32 * u + l);
      for (int k = 128; k < c; k += 32) pair(row[k / 2 + l], k + l);
    }

    // Density pass: posf by slot; ENERGY: eatom by atom (FP64 densities and pair energies).
    template <bool MULTI, bool ENERGY, bool MIX>
    __global__ __launch_bounds__(TT) void k_tile_density(EAMTables const* __restrict__ Tp, Shifts S, TileArgs A, double4* __restrict__ posf,
                                                         double* __restrict__ eatom, unsigned* __restrict__ err) {
      EAMTables const& T = *Tp;
      extern __shared__ double2 s_stage[];
      double2* const xy = s_stage;
      double2* const zw = s_stage + A.cap;
      __shared__ TileLds L;
      __shared__ SplineDesc s_phi[MULTI ? MAX_TYPES * MAX_TYPES : 1], s_V[MULTI && ENERGY ? MAX_TYPES * MAX_TYPES : 1];
      if (MULTI && threadIdx.x < T.ntypes * T.ntypes) {
        s_phi[threadIdx.x] = T.phi[threadIdx.x];
        if (ENERGY) s_V[threadIdx.x] = T.V[threadIdx.x];
      }
      unsigned e = 0;
      stage_tile(A, S, L, xy, zw, [](int, unsigned) {});
      int const rows = L.oo[16];
      int const l = threadIdx.x & 15;
      // Four rows a wavefront; its lanes stay together (walk_tile_grouped reads across them): lanes without a
      // row get the last one with no entries.
      for (int r0 = (threadIdx.x >> 6) * 4; r0 < rows; r0 += TT / 16) {
        int const r = r0 + static_cast<int>((threadIdx.x & 63) >> 4);
        int const rr = min(r, rows - 1);
        int const q = line_of(L.oo, rr);
        long const i = L.os[q] + (rr - L.oo[q]);
        double4 const pi = A.pos[i];
        int const ti = MULTI ? checked_type(static_cast<uint32_t>(pi.w), T.ntypes, e) : A.t0;
        int const c = r < rows ? min(A.cnt[i], A.K) : 0;
        double rho = 0.0, vs = 0.0;
        auto phi_of = [&](double w) -> SplineDesc const& {
          int const tj = MULTI ? checked_type(static_cast<uint32_t>(w), T.ntypes, e) : A.t0;
          return MULTI ? s_phi[tj + T.ntypes * ti] : T.phi[tj + T.ntypes * ti];
        };
        if constexpr (MIX && !ENERGY) {
          walk_tile_grouped(A.rows + i * A.rowW, c, l, pi, T.rc2, xy, zw, [&](auto const& G) {
            constexpr int NB = sizeof(G.in) / sizeof(bool);
            Seg<true> g[NB];
            float4 co[NB];
#pragma unroll
            for (int n = 0; n < NB; ++n) {
              SplineDesc const& sp = phi_of(G.p[n].w);
              float const r2f = G.in[n] ? static_cast<float>(G.p[n].r2) : 1.0f;
              g[n] = seg_of<true>(sp, r2f * __frsqrt_rn(r2f), G.in[n], e);
              co[n] = coef_of<true>(T, sp, g[n]);
            }
#pragma unroll
            for (int n = 0; n < NB; ++n) {
              double const f = static_cast<double>(poly0(co[n], g[n].t));
              rho = g[n].use ? __dadd_rn(rho, f) : rho;
            }
          });
        } else {
          walk_tile(A.rows + i * A.rowW, c, l, pi, T.rc2, xy, zw, [&](PairGeo const& p) {
            double const d = sqrt(p.r2);
            rho = __dadd_rn(rho, spl64<0>(T, phi_of(p.w), d, e));
            if (ENERGY) {
              int const tj = MULTI ? checked_type(static_cast<uint32_t>(p.w), T.ntypes, e) : A.t0;
              vs = __dadd_rn(vs, spl64<0>(T, MULTI ? s_V[vidx(T, ti, tj)] : T.V[vidx(T, ti, tj)], d, e));
            }
          });
        }
        rho = total16(rho);
        if (ENERGY) vs = total16(vs);
        if (l == 0 && r < rows) {
          posf[i] = make_double4(pi.x, pi.y, pi.z, rho);
          if (ENERGY) eatom[A.order[i]] = vs;
        }
      }
      // The embedding spline once per row and thread, instead of by one lane in 16 beside the walks.
      __syncthreads();
      for (int r = threadIdx.x; r < rows; r += TT) {
        int const q = line_of(L.oo, r);
        long const i = L.os[q] + (r - L.oo[q]);
        int const ti = MULTI ? checked_type(A.types[i], T.ntypes, e) : A.t0;
        double f, fp;
        spl64_ffp(T, T.F[ti], posf[i].w, f, fp, e);
        posf[i].w = MIX && !ENERGY ? pack_fp_type(static_cast<float>(fp), ti) : fp;
        if (ENERGY) {
          int const a = A.order[i];
          eatom[a] = 0.5 * eatom[a] + f;
        }
      }
      if (e) atomicOr(err, e);
    }

    template <bool MULTI, bool MIX>
    __global__ __launch_bounds__(TT) void k_tile_force(EAMTables const* __restrict__ Tp, Shifts S, TileArgs A, double* __restrict__ grad,
                                                       unsigned* __restrict__ err) {
      EAMTables const& T = *Tp;
      extern __shared__ double2 s_stage[];
      double2* const xy = s_stage;
      double2* const zw = s_stage + A.cap;
      uint8_t* const typ = reinterpret_cast<uint8_t*>(zw + A.cap);   // FP64 with several species
      __shared__ TileLds L;
      __shared__ SplineDesc s_phi[MULTI ? MAX_TYPES * MAX_TYPES : 1], s_V[MULTI ? MAX_TYPES * MAX_TYPES : 1];
      if (MULTI && threadIdx.x < T.ntypes * T.ntypes) {
        s_phi[threadIdx.x] = T.phi[threadIdx.x];
        s_V[threadIdx.x] = T.V[threadIdx.x];
      }
      unsigned e = 0;
      stage_tile(A, S, L, xy, zw, [&](int k, unsigned slot) {
        if (MULTI && !MIX) typ[k] = static_cast<uint8_t>(checked_type(A.types[slot], T.ntypes, e));
      });
      int const rows = L.oo[16];
      int const l = threadIdx.x & 15;
      for (int r = threadIdx.x >> 4; r < rows; r += TT / 16) {
        int const q = line_of(L.oo, r);
        long const i = L.os[q] + (r - L.oo[q]);
        int const ia = A.order[i];
        double4 const pi = A.pos[i];
        int const c = min(A.cnt[i], A.K);
        // Mixed form: the species the density pass packed beside F' (checked there).
        int const ti = MULTI ? (MIX ? packed_type(pi.w) : checked_type(A.types[i], T.ntypes, e)) : A.t0;
        bool const act = !A.frozen[ia];
        double gx = 0.0, gy = 0.0, gz = 0.0;
        walk_tile(A.rows + i * A.rowW, act ? c : 0, l, pi, T.rc2, xy, zw, [&](PairGeo const& p) {
          int const tj = MULTI ? (MIX ? packed_type(p.w) : typ[p.j]) : A.t0;
          SplineDesc const& sv = MULTI ? s_V[vidx(T, ti, tj)] : T.V[vidx(T, ti, tj)];
          SplineDesc const& sa = MULTI ? s_phi[tj + T.ntypes * ti] : T.phi[tj + T.ntypes * ti];
          double cf;
          if (MIX) {
            float r2f = static_cast<float>(p.r2);
            float rinv = __frsqrt_rn(r2f);
            float rf = r2f * rinv;
            float vp = spl32f<1>(T, sv, rf, e);
            float pa = spl32f<1>(T, sa, rf, e);
            // phi_{g->a} is phi_{a->g} for a same-species pair: no second table load.
            float pb = MULTI && ti != tj ? spl32f<1>(T, s_phi[MULTI ? ti + T.ntypes * tj : 0], rf, e) : pa;
            float mag = vp + packed_fp(pi.w) * pa + packed_fp(p.w) * pb;
            cf = static_cast<double>(mag * rinv);
          } else {
            double d = sqrt(p.r2);
            double vp = spl64<1>(T, sv, d, e);
            double pa = spl64<1>(T, sa, d, e);
            double pb = MULTI && ti != tj ? spl64<1>(T, s_phi[MULTI ? ti + T.ntypes * tj : 0], d, e) : pa;
            cf = (vp + pi.w * pa + p.w * pb) / d;
          }
          gx = __dadd_rn(gx, -cf * p.dx);
          gy = __dadd_rn(gy, -cf * p.dy);
          gz = __dadd_rn(gz, -cf * p.dz);
        });
        gx = total16(gx);
        gy = total16(gy);
        gz = total16(gz);
        if (l < 3) grad[3l * ia + l] = act ? (l == 0 ? gx : (l == 1 ? gy : gz)) : 0.0;
      }
      if (e) atomicOr(err, e);
    }

    // ---- Hessian-vector product ---------------------------------------------------------------------
    // One reciprocal and one segment fetch per table and pair; rows from the plain list (L lanes an atom, small
    // systems) or tile by tile with positions, the masked direction v and (F', dF') staged in LDS, where
    // a pair takes no gather but its table segments (row gathers: 51 + 122 us at 54.5k atoms).

    struct HvpSum {
      double x = 0, y = 0, z = 0;
    };

    __device__ inline void hvp_density_pair(EAMTables const& T, SplineDesc const& sa, double dx, double dy, double dz, double r2,
                                            double vx, double vy, double vz, double& rho, double& drho, unsigned& e) {
      double const r = sqrt(r2);
      double f, fp;
      spl64_ffp(T, sa, r, f, fp, e);
      rho += f;
      drho += fp * ((dx * vx + dy * vy + dz * vz) / r);
    }

    // dv = v_a - v_g, (F', dF') of the row's atom (di) and of the neighbour (dj).
    template <bool MULTI>
    __device__ inline void hvp_force_pair(EAMTables const& T, SplineDesc const& sv, SplineDesc const& sa, SplineDesc const& sb,
                                          bool same, double dx, double dy, double dz, double r2, double vx, double vy,
                                          double vz, double2 di, double2 dj, HvpSum& h, unsigned& e) {
      double const r = sqrt(r2), inv = 1.0 / r;
      double const ux = dx * inv, uy = dy * inv, uz = dz * inv;
      double const s = ux * vx + uy * vy + uz * vz;
      double vp, vpp, pa, paa;
      spl64_12(T, sv, r, vp, vpp, e);
      spl64_12(T, sa, r, pa, paa, e);   // phi_{a->g}
      double pb = pa, pbb = paa;        // phi_{g->a}
      if (MULTI && !same) spl64_12(T, sb, r, pb, pbb, e);
      double const m = vp + di.x * pa + dj.x * pb;
      double const dm = (vpp + di.x * paa + dj.x * pbb) * s + di.y * pa + dj.y * pb;
      double const q = m * inv;
      h.x -= dm * ux + q * (vx - ux * s);
      h.y -= dm * uy + q * (vy - uy * s);
      h.z -= dm * uz + q * (vz - uz * s);
    }

    template <int L, bool MULTI>
    __global__ __launch_bounds__(NT) void k_hvp_density(EAMTables const* __restrict__ Tp, Shifts S, PairArgs A, double const* __restrict__ v,
                                                        double2* __restrict__ dfp, unsigned* __restrict__ err) {
      EAMTables const& T = *Tp;
      long gid = xcd_block(blockIdx.x, gridDim.x) * static_cast<long>(NT) + threadIdx.x;
      long i = gid / L;
      int lane = static_cast<int>(gid % L);
      bool act = i < A.n;
      double rho = 0, drho = 0;
      unsigned e = 0;
      int ti = 0;
      if (act) {
        double4 pi = A.pos[i];
        ti = MULTI ? checked_type(A.types[i], T.ntypes, e) : A.t0;
        bool fi = A.frozen[i];
        double vix = fi ? 0 : v[3 * i], viy = fi ? 0 : v[3 * i + 1], viz = fi ? 0 : v[3 * i + 2];
        int const c = min(A.cnt[i], A.K);
        unsigned const* row = A.nbr + i * static_cast<long>(A.K);
        for (int k = lane; k < c; k += L) {
          PairGeo const p = geo(S, A.pos, row[k], pi);
          long const j = p.j;
          bool const fj = A.frozen[j];
          double vjx = fj ? 0 : v[3 * j], vjy = fj ? 0 : v[3 * j + 1], vjz = fj ? 0 : v[3 * j + 2];
          int tj = MULTI ? checked_type(A.types[j], T.ntypes, e) : A.t0;
          if (p.r2 < T.rc2)
            hvp_density_pair(T, T.phi[tj + T.ntypes * ti], p.dx, p.dy, p.dz, p.r2, vjx - vix, vjy - viy, vjz - viz, rho, drho, e);
        }
      }
      rho = group_sum<L>(rho);
      drho = group_sum<L>(drho);
      if (act && lane == 0) {
        double fp, fpp;
        spl64_12(T, T.F[ti], rho, fp, fpp, e);
        dfp[i] = make_double2(fp, fpp * drho);
      }
      if (e) atomicOr(err, e);
    }

    template <int L, bool MULTI>
    __global__ __launch_bounds__(NT) void k_hvp_force(EAMTables const* __restrict__ Tp, Shifts S, PairArgs A, double const* __restrict__ v,
                                                      double2 const* __restrict__ dfp, double* __restrict__ hv,
                                                      unsigned* __restrict__ err) {
      EAMTables const& T = *Tp;
      long gid = xcd_block(blockIdx.x, gridDim.x) * static_cast<long>(NT) + threadIdx.x;
      long i = gid / L;
      int lane = static_cast<int>(gid % L);
      bool inr = i < A.n;
      bool act = inr && !A.frozen[i];
      HvpSum h;
      unsigned e = 0;
      if (act) {
        double4 pi = A.pos[i];
        double2 di = dfp[i];
        int ti = MULTI ? checked_type(A.types[i], T.ntypes, e) : A.t0;
        double vix = v[3 * i], viy = v[3 * i + 1], viz = v[3 * i + 2];
        int const c = min(A.cnt[i], A.K);
        unsigned const* row = A.nbr + i * static_cast<long>(A.K);
        for (int k = lane; k < c; k += L) {
          PairGeo const p = geo(S, A.pos, row[k], pi);
          long const j = p.j;
          bool const fj = A.frozen[j];
          double vjx = fj ? 0 : v[3 * j], vjy = fj ? 0 : v[3 * j + 1], vjz = fj ? 0 : v[3 * j + 2];
          double2 const dj = dfp[j];
          int tj = MULTI ? checked_type(A.types[j], T.ntypes, e) : A.t0;
          if (p.r2 < T.rc2)
            hvp_force_pair<MULTI>(T, T.V[vidx(T, ti, tj)], T.phi[tj + T.ntypes * ti], T.phi[ti + T.ntypes * tj], ti == tj, p.dx,
                                  p.dy, p.dz, p.r2, vjx - vix, vjy - viy, vjz - viz, di, dj, h, e);
        }
      }
      h.x = group_sum<L>(h.x);
      h.y = group_sum<L>(h.y);
      h.z = group_sum<L>(h.z);
      if (inr && lane < 3) hv[3 * i + lane] = act ? (lane == 0 ? h.x : (lane == 1 ? h.y : h.z)) : 0.0;
      if (e) atomicOr(err, e);
    }

    // Tiled passes: the stage holds (x, y), (z, vz), (vx, vy) and, in the force pass, (F', dF') of every entry, and its
    // species with several.  dfp by slot.
    template <bool MULTI, bool FORCE>
    __global__ __launch_bounds__(TT) void k_tile_hvp(EAMTables const* __restrict__ Tp, Shifts S, TileArgs A, double const* __restrict__ v,
                                                     double2* __restrict__ dfp, double* __restrict__ hv,
                                                     unsigned* __restrict__ err) {
      EAMTables const& T = *Tp;
      extern __shared__ double2 s_stage[];
      double2* const xy = s_stage;
      double2* const zv = xy + A.cap;
      double2* const vv = zv + A.cap;
      double2* const df = vv + A.cap;
      uint8_t* const typ = reinterpret_cast<uint8_t*>(df + (FORCE ? A.cap : 0));
      __shared__ TileLds L;
      __shared__ SplineDesc s_phi[MULTI ? MAX_TYPES * MAX_TYPES : 1], s_V[MULTI && FORCE ? MAX_TYPES * MAX_TYPES : 1];
      if (MULTI && threadIdx.x < T.ntypes * T.ntypes) {
        s_phi[threadIdx.x] = T.phi[threadIdx.x];
        if (FORCE) s_V[threadIdx.x] = T.V[threadIdx.x];
      }
      unsigned e = 0;
      stage_tile(A, S, L, xy, zv, [&](int k, unsigned slot) {
        long const a = A.order[slot];
        bool const f = A.frozen[a];
        vv[k] = make_double2(f ? 0 : v[3 * a], f ? 0 : v[3 * a + 1]);
        zv[k].y = f ? 0 : v[3 * a + 2];
        if (FORCE) df[k] = dfp[slot];
        if (MULTI) typ[k] = static_cast<uint8_t>(checked_type(A.types[slot], T.ntypes, e));
      });
      int const rows = L.oo[16];
      int const l = threadIdx.x & 15;
      for (int r = threadIdx.x >> 4; r < rows; r += TT / 16) {
        int const q = line_of(L.oo, r);
        long const i = L.os[q] + (r - L.oo[q]);
        long const ia = A.order[i];
        double4 const pi = A.pos[i];
        int const c = min(A.cnt[i], A.K);
        int const ti = MULTI ? checked_type(A.types[i], T.ntypes, e) : A.t0;
        bool const fi = A.frozen[ia];
        double const vix = fi ? 0 : v[3 * ia], viy = fi ? 0 : v[3 * ia + 1], viz = fi ? 0 : v[3 * ia + 2];
        double2 const di = FORCE ? dfp[i] : make_double2(0, 0);
        double rho = 0, drho = 0;
        HvpSum h;
        walk_tile(A.rows + i * A.rowW, FORCE && fi ? 0 : c, l, pi, T.rc2, xy, zv, [&](PairGeo const& p) {
          double2 const w = vv[p.j];
          int const tj = MULTI ? typ[p.j] : A.t0;
          SplineDesc const& sa = MULTI ? s_phi[tj + T.ntypes * ti] : T.phi[tj + T.ntypes * ti];
          if constexpr (FORCE) {
            SplineDesc const& sv = MULTI ? s_V[vidx(T, ti, tj)] : T.V[vidx(T, ti, tj)];
            hvp_force_pair<MULTI>(T, sv, sa, s_phi[MULTI ? ti + T.ntypes * tj : 0], ti == tj, p.dx, p.dy, p.dz, p.r2, w.x - vix,
                                  w.y - viy, p.w - viz, di, df[p.j], h, e);
          } else {
            hvp_density_pair(T, sa, p.dx, p.dy, p.dz, p.r2, w.x - vix, w.y - viy, p.w - viz, rho, drho, e);
          }
        });
        if constexpr (FORCE) {
          double const hx = total16(h.x), hy = total16(h.y), hz = total16(h.z);
          if (l < 3) hv[3 * ia + l] = fi ? 0.0 : (l == 0 ? hx : (l == 1 ? hy : hz));
        } else {
          rho = total16(rho);
          drho = total16(drho);
          if (l == 0) dfp[i] = make_double2(rho, drho);
        }
      }
      if constexpr (!FORCE) {   // the embedding spline, a row a thread
        __syncthreads();
        for (int r = threadIdx.x; r < rows; r += TT) {
          int const q = line_of(L.oo, r);
          long const i = L.os[q] + (r - L.oo[q]);
          int const ti = MULTI ? checked_type(A.types[i], T.ntypes, e) : A.t0;
          double2 const d = dfp[i];
          double fp, fpp;
          spl64_12(T, T.F[ti], d.x, fp, fpp, e);
          dfp[i] = make_double2(fp, fpp * d.y);
        }
      }
      if (e) atomicOr(err, e);
    }

    // FP64 densities only (base state of batched searches).
    template <int L, bool MULTI>
    __global__ __launch_bounds__(NT) void k_rho(EAMTables const* __restrict__ Tp, Shifts S, PairArgs A, double* __restrict__ rho_out,
                                                unsigned* __restrict__ err) {
      EAMTables const& T = *Tp;
      long gid = xcd_block(blockIdx.x, gridDim.x) * static_cast<long>(NT) + threadIdx.x;
      long i = gid / L;
      int lane = static_cast<int>(gid % L);
      bool act = i < A.n;
      double rho = 0;
      unsigned e = 0;
      if (act) {
        double4 pi = A.pos[i];
        int ti = MULTI ? checked_type(A.types[i], T.ntypes, e) : A.t0;
        int const c = min(A.cnt[i], A.K);
        unsigned const* row = A.nbr + i * static_cast<long>(A.K);
        for (int k = lane; k < c; k += L) {
          unsigned en = row[k];
          unsigned j = en & NB_IDX_MASK;
          double3 sh = S.of(en >> NB_SHIFT_BITS);
          double4 pj = A.pos[j];
          double dx = (pj.x + sh.x) - pi.x, dy = (pj.y + sh.y) - pi.y, dz = (pj.z + sh.z) - pi.z;
          double r2 = dx * dx + dy * dy + dz * dz;
          if (r2 < T.rc2) {
            int tj = MULTI ? checked_type(A.types[j], T.ntypes, e) : A.t0;
            rho += spl64<0>(T, T.phi[tj + T.ntypes * ti], sqrt(r2), e);
          }
        }
      }
      rho = group_sum<L>(rho);
      if (act && lane == 0) rho_out[i] = rho;
      if (e) atomicOr(err, e);
    }

    __global__ void k_table_eval(EAMTables T, SplineDesc s, double const* __restrict__ x, long m, int deriv,
                                 double* __restrict__ out, unsigned* __restrict__ err) {
      long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
      if (i >= m) return;
      unsigned e = 0;
      double v = deriv == 0 ? spl64<0>(T, s, x[i], e) : deriv == 1 ? spl64<1>(T, s, x[i], e) : spl64<2>(T, s, x[i], e);
      out[i] = v;
      if (e) atomicOr(err, e);
    }

    __global__ void k_types_by_slot(uint32_t const* __restrict__ types, int const* __restrict__ order, long n,
                                    uint32_t* __restrict__ out, double4* __restrict__ gpos) {
      long k = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
      if (k < n) {
        uint32_t const t = types[order[k]];
        out[k] = t;
        gpos[k].w = static_cast<double>(t);
      }
    }

    // The gradient and energy passes run in the list's slot (cell) order: a workgroup's atoms are neighbours in
    // space and so are the rows they read.  With several species the types are gathered into slot order, and into the
    // w slot of the slot-ordered positions (the density pass reads a neighbour's species from there): once per list
    // build for staged host types (the library sees every change of them), on every call for device types.  Type
    // stamps are unique across handles, so a list shared by several potentials or type arrays is re-gathered
    // whenever another one wrote its w slots last.
    uint32_t const* types_by_slot(flyg_eam_s& E, flyg_list_s& nl, uint32_t const* types) {
      bool const staged = types == E.types.get();
      bool const cached = staged && E.gtype_build == nl.build_id && E.gtype_stamp == E.types_stamp &&
                          nl.wtype_build == nl.build_id && nl.wtype_stamp == E.types_stamp;
      if (!cached) {
        E.gtype_build = -1;   // the buffer may be reallocated: its contents are no longer known
        nl.wtype_build = -1;
        E.gtype.reserve(nl.n);
        k_types_by_slot<<<static_cast<unsigned>((nl.n + 255) / 256), 256, 0, E.ctx->stream>>>(
            types, nl.order.get(), nl.n, E.gtype.get(), nl.gpos.get());
        HIPCHK(hipGetLastError());
        if (staged) {
          E.gtype_build = nl.build_id;
          E.gtype_stamp = E.types_stamp;
          nl.wtype_build = nl.build_id;
          nl.wtype_stamp = E.types_stamp;
        }
      }
      return E.gtype.get();
    }

    // nbr in slot order, entries naming slots.
    __global__ __launch_bounds__(NT) void k_slot_rows(unsigned const* __restrict__ nbr, int const* __restrict__ gcnt,
                                                      int const* __restrict__ order, int const* __restrict__ rank, int K,
                                                      long n, unsigned* __restrict__ out) {
      long const gid = xcd_block(blockIdx.x, gridDim.x) * static_cast<long>(NT) + threadIdx.x, i = gid / 16;
      if (i >= n) return;
      unsigned const* row = nbr + order[i] * static_cast<long>(K);
      int const c = min(gcnt[i], K);
      for (int k = static_cast<int>(gid % 16); k < c; k += 16) {
        unsigned const en = row[k];
        out[i * K + k] = (en & ~NB_IDX_MASK) | static_cast<unsigned>(rank[en & NB_IDX_MASK]);
      }
    }

    unsigned grid_for(long n, int L) { return static_cast<unsigned>((n * L + NT - 1) / NT); }

    // A tiled list keeps its plain rows by atom.  Atoms far apart in space then share a workgroup, and with atoms in no
    // spatial order every gather is a cache line of its own: 116 us a gradient (two species, FP64, 54.5k atoms
    // shuffled, 8 lanes) where rows in slot order take 64.  They are made once per build, in 8 us.  A captured
    // call walks the rows by atom: a graph launched after a rebuild must not find the last build's copy.
    bool slot_rows(flyg_eam_s& E, flyg_list_s& nl) {
      hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
      HIPCHK(hipStreamIsCapturing(E.ctx->stream, &st));
      if (st != hipStreamCaptureStatusNone) return false;
      if (nl.srows_build == nl.build_id) return true;
      nl.srows.reserve(static_cast<std::size_t>(nl.n) * nl.K);
      k_slot_rows<<<grid_for(nl.n, 16), NT, 0, E.ctx->stream>>>(nl.nbr.get(), nl.gcnt.get(), nl.order.get(), nl.rank.get(),
                                                                nl.K, nl.n, nl.srows.get());
      HIPCHK(hipGetLastError());
      nl.srows_build = nl.build_id;
      return true;
    }

    // Plain rows in slot order.
    PairArgs slot_args(flyg_eam_s& E, flyg_list_s& nl, uint32_t const* types, uint8_t const* frozen) {
      PairArgs A = pair_args(E, nl, types, frozen);
      if (nl.tiled && !slot_rows(E, nl)) return A;
      A.pos = nl.gpos.get();
      A.nbr = nl.tiled ? nl.srows.get() : nl.rows.get();
      A.cnt = nl.gcnt.get();
      A.order = nl.order.get();
      if (A.t0 < 0) {
        A.types = types_by_slot(E, nl, types);
        A.type_in_w = true;
      }
      return A;
    }

    TileArgs tile_args(flyg_eam_s& E, flyg_list_s& nl, uint32_t const* types, uint8_t const* frozen) {
      PairArgs const P = pair_args(E, nl, types, frozen);
      TileArgs A{nl.tile,        nl.cstart.get(), nl.sslot.get(), nl.rows.get(), nl.rowK / 2, nl.K, nl.gcnt.get(),
                 nl.order.get(), nl.gpos.get(),   nullptr,        frozen,        P.t0,        0};
      A.cap = (nl.tile_most + 15) & ~15;
      if (A.t0 < 0) A.types = types_by_slot(E, nl, types);
      return A;
    }

    // Lanes per atom for the base densities of batched searches.
    constexpr int LANES = 8;

  }  // namespace

  void eam_setup_tables(flyg_eam_s& E) {
    SetflData const& D = E.data;
    int const n = D.ntypes;
    std::vector<double4> all;
    EAMTables T{};
    T.ntypes = n;
    T.rc = D.rcut;
    T.rc2 = D.rcut * D.rcut;
    T.rcf = static_cast<float>(D.rcut);
    auto add = [&](std::vector<double> const& y, double dx) {
      std::vector<double4> c = spline_coefficients(y, dx);
      SplineDesc s{};
      s.off = static_cast<int>(all.size());
      s.count = static_cast<int>(c.size());
      s.dx = dx;
      s.inv_dx = 1 / dx;
      s.dxf = static_cast<float>(dx);
      s.inv_dxf = static_cast<float>(1 / dx);
      all.insert(all.end(), c.begin(), c.end());
      return s;
    };
    for (int a = 0; a < n; ++a) T.F[a] = add(D.F[a], D.drho);
    for (int k = 0; k < n * n; ++k) T.phi[k] = add(D.phi[k], D.dr);
    for (int a = 0; a < n; ++a)
      for (int b = 0; b <= a; ++b) T.V[a + n * b] = add(D.V[a + n * b], D.dr);
    std::vector<float4> all32(all.size());
    for (std::size_t i = 0; i < all.size(); ++i)
      all32[i] = make_float4(static_cast<float>(all[i].x), static_cast<float>(all[i].y), static_cast<float>(all[i].z),
                             static_cast<float>(all[i].w));
    E.c64.reserve(all.size());
    E.c32.reserve(all.size());
    HIPCHK(hipMemcpy(E.c64.get(), all.data(), all.size() * sizeof(double4), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(E.c32.get(), all32.data(), all32.size() * sizeof(float4), hipMemcpyHostToDevice));
    T.c64 = E.c64.get();
    T.c32 = E.c32.get();
    E.tab = T;
    E.dtab.reserve(1);
    HIPCHK(hipMemcpy(E.dtab.get(), &E.tab, sizeof(EAMTables), hipMemcpyHostToDevice));
  }

  namespace {
    // energy = true: FP64 densities and pair energies (energies are always FP64); otherwise the density
    // pass of a gradient in the given precision.
    template <int L>
    void launch_density(flyg_eam_s& E, Shifts const& S, PairArgs const& A, bool energy, int precision, double4* pf) {
      hipStream_t st = E.ctx->stream;
      unsigned* err = E.ctx->dflags.get();
      bool multi = A.t0 < 0;
      bool mix = precision == FLYG_MIXED;
      unsigned g = grid_for(A.n, L);
      if (multi) {
        if (energy)
          k_density<L, true, true, false><<<g, NT, 0, st>>>(E.dtab.get(), S, A, pf, E.eatom.get(), err);
        else if (mix)
          k_density<L, true, false, true><<<g, NT, 0, st>>>(E.dtab.get(), S, A, pf, nullptr, err);
        else
          k_density<L, true, false, false><<<g, NT, 0, st>>>(E.dtab.get(), S, A, pf, nullptr, err);
      } else {
        if (energy)
          k_density<L, false, true, false><<<g, NT, 0, st>>>(E.dtab.get(), S, A, pf, E.eatom.get(), err);
        else if (mix)
          k_density<L, false, false, true><<<g, NT, 0, st>>>(E.dtab.get(), S, A, pf, nullptr, err);
        else
          k_density<L, false, false, false><<<g, NT, 0, st>>>(E.dtab.get(), S, A, pf, nullptr, err);
      }
    }

    template <int L>
    void launch_force(flyg_eam_s& E, Shifts const& S, PairArgs const& A, double* grad, int precision,
                      double4 const* pf) {
      hipStream_t st = E.ctx->stream;
      unsigned* err = E.ctx->dflags.get();
      bool multi = A.t0 < 0;
      bool mix = precision == FLYG_MIXED;
      unsigned g = grid_for(A.n, L);
      if (multi) {
        if (mix)
          k_force<L, true, true><<<g, NT, 0, st>>>(E.dtab.get(), S, A, pf, grad, err);
        else
          k_force<L, true, false><<<g, NT, 0, st>>>(E.dtab.get(), S, A, pf, grad, err);
      } else {
        if (mix)
          k_force<L, false, true><<<g, NT, 0, st>>>(E.dtab.get(), S, A, pf, grad, err);
        else
          k_force<L, false, false><<<g, NT, 0, st>>>(E.dtab.get(), S, A, pf, grad, err);
      }
    }
  }  // namespace

  namespace {
    void tile_density(flyg_eam_s& E, Shifts const& S, TileArgs const& A, bool energy, int precision, double4* pf) {
      unsigned const g = static_cast<unsigned>(A.G.ntiles);
      std::size_t const lds = static_cast<std::size_t>(A.cap) * sizeof(double4);
      unsigned* err = E.ctx->dflags.get();
      auto run = [&](auto k) { k<<<g, TT, lds, E.ctx->stream>>>(E.dtab.get(), S, A, pf, E.eatom.get(), err); };
      bool const mix = precision == FLYG_MIXED;
      if (A.t0 < 0) {
        energy ? run(k_tile_density<true, true, false>)
               : (mix ? run(k_tile_density<true, false, true>) : run(k_tile_density<true, false, false>));
      } else {
        energy ? run(k_tile_density<false, true, false>)
               : (mix ? run(k_tile_density<false, false, true>) : run(k_tile_density<false, false, false>));
      }
    }

    void tile_force(flyg_eam_s& E, Shifts const& S, TileArgs const& A, double* grad, int precision) {
      unsigned const g = static_cast<unsigned>(A.G.ntiles);
      bool const mix = precision == FLYG_MIXED;
      std::size_t const lds = static_cast<std::size_t>(A.cap) * (sizeof(double4) + (A.t0 < 0 && !mix ? 1 : 0));
      auto run = [&](auto k) { k<<<g, TT, lds, E.ctx->stream>>>(E.dtab.get(), S, A, grad, E.ctx->dflags.get()); };
      if (A.t0 < 0) {
        mix ? run(k_tile_force<true, true>) : run(k_tile_force<true, false>);
      } else {
        mix ? run(k_tile_force<false, true>) : run(k_tile_force<false, false>);
      }
    }
  }  // namespace

  double eam_energy(flyg_eam_s& E, flyg_list_s& nl, uint32_t const* types, uint8_t const* frozen) {
    require(nl.built, "List used before rebuild");
    require(E.tab.rc <= nl.rc, "r_cut is bigger than the internal r_cut of the list");
    E.posf.reserve(nl.n);
    E.eatom.reserve(nl.n);
    Shifts const S = shifts_of(nl.box);
    if (nl.tiled && E.lanes <= 0) {
      tile_density(E, S, tile_args(E, nl, types, frozen), true, FLYG_FP64, E.posf.get());
    } else {
      launch_density<16>(E, S, slot_args(E, nl, types, frozen), true, FLYG_FP64, E.posf.get());
    }
    HIPCHK(hipGetLastError());
    dev_sum(*E.ctx, E.eatom.get(), nl.n, E.ctx->hpart, E.ctx->hflags + 1);
    HIPCHK(hipStreamSynchronize(E.ctx->stream));
    if (E.ctx->hflags[1]) throw_flags(E.ctx->take_flags());
    return host_sum(E.ctx->hpart, 0, nl.n);
  }

  namespace {
    // Density then force pass; pf holds the pass-1 output (positions + F') of every atom.
    void density_with(flyg_eam_s& E, Shifts const& S, PairArgs const& A, int precision, int L, double4* pf) {
      switch (L) {
        case 4:
          launch_density<4>(E, S, A, false, precision, pf);
          break;
        case 16:
          launch_density<16>(E, S, A, false, precision, pf);
          break;
        default:
          launch_density<8>(E, S, A, false, precision, pf);
      }
    }

    void force_with(flyg_eam_s& E, Shifts const& S, PairArgs const& A, double* d_grad, int precision, int L,
                    double4 const* pf) {
      switch (L) {
        case 4:
          launch_force<4>(E, S, A, d_grad, precision, pf);
          break;
        case 16:
          launch_force<16>(E, S, A, d_grad, precision, pf);
          break;
        default:
          launch_force<8>(E, S, A, d_grad, precision, pf);
      }
    }

    // Lanes per atom row of the plain-row passes.  The row sums do not depend on them (Acc16).  16 unless the handle
    // names a count: more lanes shorten each row's chain of dependent gathers, which is what bounds the sizes left to
    // these passes.  Density / force, us, FP64 at 16, 8 and 4 lanes: 8.2k atoms 6.6/8.1, 9.6/11.5, 13.4/17.8; 16k
    // 9.4/10.2, 8.5/13.4, 11.3/14.8.  Timing the three counts on a potential's first call cost 24 launches and
    // could keep a slower one.  Eight lanes where 16 would take a second, nearly empty round of workgroups (2048 of
    // 256 threads are resident, in the FP64 form with its registers fewer).  16 / 8 lanes, two species, list cut-offs
    // 5.5 / 6.8 A: mixed 31k atoms 26.5/25.7 34.9/36.3, 35k 31.6/28.5 45.2/40.4, 44k 35.6/33.7 59.6/53.6, 54k equal;
    // FP64 28k 33.0/33.2 40.9/44.6, 31k 37.9/33.1 50.8/45.6, 39k 44.2/40.1 65.8/58.8, 44k 47.9/48.7 74.9/69.9.
    // Fewer also where a dilute system's rows would leave most of 16 idle, 16 / 8 / 4 lanes, mixed, 216k atoms with rows
    // of 4, 8, 17, 34, 46: 43/28/25, 51/32/31, 79/50/49, 84/72/81, 91/95/99; 33k: 11/10/10, 12/11/10, 16/13/14,
    // 17/16/22, 18/19/26; below 20k they are equal.
    void gradient_with(flyg_eam_s& E, Shifts const& S, PairArgs const& A, double row, double* d_grad, int precision,
                       double4* pf) {
      bool const eight = (precision == FLYG_MIXED ? A.n > 32768 && A.n < 46000 : A.n >= 30000 && A.n < 41000) ||
                         (A.n >= 20000 && row < 40.0);
      int const L = E.lanes > 0 ? E.lanes : (A.n >= 20000 && row < 7.0 ? 4 : (eight ? 8 : 16));
      density_with(E, S, A, precision, L, pf);
      force_with(E, S, A, d_grad, precision, L, pf);
    }
  }  // namespace

  void eam_gradient(flyg_eam_s& E, flyg_list_s& nl, uint32_t const* types, uint8_t const* frozen, double* d_grad,
                    int precision) {
    require(nl.built, "List used before rebuild");
    require(E.tab.rc <= nl.rc, "r_cut is bigger than the internal r_cut of the list");
    E.posf.reserve(nl.n);
    Shifts S = shifts_of(nl.box);
    if (E.timing) {   // the pair covers the species gather too
      if (E.events_used == E.events.size()) {
        hipEvent_t a, b;
        HIPCHK(hipEventCreate(&a));
        HIPCHK(hipEventCreate(&b));
        E.events.emplace_back(a, b);
      }
      HIPCHK(hipEventRecord(E.events[E.events_used].first, E.ctx->stream));
    }
    bool tiles = nl.tiled && E.lanes <= 0;
    if (tiles && nl.grad_rows && nl.grad_build == nl.build_id) tiles = !slot_rows(E, nl);
    nl.grad_build = nl.build_id;
    if (tiles) {
      TileArgs A = tile_args(E, nl, types, frozen);
      tile_density(E, S, A, false, precision, E.posf.get());
      A.pos = E.posf.get();
      tile_force(E, S, A, d_grad, precision);
    } else {
      gradient_with(E, S, slot_args(E, nl, types, frozen), nl.mean_row, d_grad, precision, E.posf.get());
    }
    if (E.timing) HIPCHK(hipEventRecord(E.events[E.events_used++].second, E.ctx->stream));
    HIPCHK(hipGetLastError());
  }

  // ---------------------------------------------------------------------------------------------------
  // Allocation-free gradient.  The pass-1 output goes to a file-scope device array instead of the
  // handle's buffer; each GPU holds its own copy of the array (at its own address, looked up once per
  // device when a context is created there) until the process ends, and every call on that GPU shares it,
  // so calls that overlap on one GPU race.  The density pass writes every entry the force pass reads, so
  // nothing needs clearing between calls.
  // ---------------------------------------------------------------------------------------------------

  namespace {
    static __device__ __align__(256) double4 scratch[NOALLOC_MAX_ATOMS];

    constexpr int MAX_DEVICES = 64;
    std::mutex g_scratch_mu;
    double4* g_scratch_ptr[MAX_DEVICES] = {};
  }  // namespace

  void noalloc_scratch_init(int device) {
    require(device >= 0 && device < MAX_DEVICES, "device index out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[device]) return;
    void* p = nullptr;
    // The array's name is a host-side stand-in; kernels get this device address (the device is current).
    HIPCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_ptr[device] = static_cast<double4*>(p);
  }

  void eam_gradient_noalloc(flyg_eam_s& E, flyg_list_s& nl, uint32_t const* d_types, uint8_t const* d_frozen,
                            double* d_grad, int precision) {
    require(nl.built, "List used before rebuild");
    require(E.tab.rc <= nl.rc, "r_cut is bigger than the internal r_cut of the list");
    require(nl.n <= NOALLOC_MAX_ATOMS, "the allocation-free gradient takes at most 131072 atoms");
    double4* pf = nullptr;
    {
      std::lock_guard<std::mutex> lock(g_scratch_mu);
      int const dev = E.ctx->device;
      if (dev >= 0 && dev < MAX_DEVICES) pf = g_scratch_ptr[dev];
    }
    require(pf != nullptr, "no scratch address for this device (its context was not created)");
    Shifts S = shifts_of(nl.box);
    PairArgs A = pair_args(E, nl, d_types, d_frozen);
    gradient_with(E, S, A, nl.mean_row, d_grad, precision, pf);
    HIPCHK(hipGetLastError());
  }

  // The largest stage of any pass fits the 160 KB of LDS a workgroup of gfx950 can have.
  static_assert((TILE_MOST + 15) / 16 * 16 * 65 + sizeof(TileLds) + 2 * MAX_TYPES * MAX_TYPES * sizeof(SplineDesc) <= 160 * 1024,
                "an HVP's stage does not fit in LDS");

  void eam_hvp(flyg_eam_s& E, flyg_list_s& nl, uint32_t const* types, uint8_t const* frozen, double const* d_v,
               double* d_hv) {
    require(nl.built, "List used before rebuild");
    require(E.tab.rc <= nl.rc, "r_cut is bigger than the internal r_cut of the list");
    E.dfp.reserve(nl.n);
    Shifts S = shifts_of(nl.box);
    hipStream_t st = E.ctx->stream;
    unsigned* err = E.ctx->dflags.get();
    if (nl.tiled && E.lanes <= 0) {
      TileArgs const A = tile_args(E, nl, types, frozen);
      unsigned const g = static_cast<unsigned>(A.G.ntiles);
      std::size_t const t = A.t0 < 0 ? 1 : 0;
      std::size_t const ld = static_cast<std::size_t>(A.cap) * (48 + t), lf = static_cast<std::size_t>(A.cap) * (64 + t);
      if (A.t0 < 0) {
        k_tile_hvp<true, false><<<g, TT, ld, st>>>(E.dtab.get(), S, A, d_v, E.dfp.get(), d_hv, err);
        k_tile_hvp<true, true><<<g, TT, lf, st>>>(E.dtab.get(), S, A, d_v, E.dfp.get(), d_hv, err);
      } else {
        k_tile_hvp<false, false><<<g, TT, ld, st>>>(E.dtab.get(), S, A, d_v, E.dfp.get(), d_hv, err);
        k_tile_hvp<false, true><<<g, TT, lf, st>>>(E.dtab.get(), S, A, d_v, E.dfp.get(), d_hv, err);
      }
      HIPCHK(hipGetLastError());
      return;
    }
    PairArgs A = pair_args(E, nl, types, frozen);
    auto rows = [&](auto lanes) {
      constexpr int L = decltype(lanes)::value;
      unsigned const g = grid_for(nl.n, L);
      if (A.t0 < 0) {
        k_hvp_density<L, true><<<g, NT, 0, st>>>(E.dtab.get(), S, A, d_v, E.dfp.get(), err);
        k_hvp_force<L, true><<<g, NT, 0, st>>>(E.dtab.get(), S, A, d_v, E.dfp.get(), d_hv, err);
      } else {
        k_hvp_density<L, false><<<g, NT, 0, st>>>(E.dtab.get(), S, A, d_v, E.dfp.get(), err);
        k_hvp_force<L, false><<<g, NT, 0, st>>>(E.dtab.get(), S, A, d_v, E.dfp.get(), d_hv, err);
      }
    };
    // Rows of a dilute system would leave most of 16 lanes idle: 216k atoms with rows of 8, 17, 25, us, 16 / 8 lanes:
    // 73/53, 122/110, 132/136.
    if (nl.mean_row < 22.0) {
      rows(std::integral_constant<int, 8>{});
    } else {
      rows(std::integral_constant<int, 16>{});
    }
    HIPCHK(hipGetLastError());
  }

  void eam_density(flyg_eam_s& E, flyg_list_s& nl, uint32_t const* d_types, double* d_rho) {
    require(nl.built, "List used before rebuild");
    Shifts S = shifts_of(nl.box);
    PairArgs A = pair_args(E, nl, d_types, nullptr);
    unsigned g = grid_for(nl.n, LANES);
    if (A.t0 < 0) {
      k_rho<LANES, true><<<g, NT, 0, E.ctx->stream>>>(E.dtab.get(), S, A, d_rho, E.ctx->dflags.get());
    } else {
      k_rho<LANES, false><<<g, NT, 0, E.ctx->stream>>>(E.dtab.get(), S, A, d_rho, E.ctx->dflags.get());
    }
    HIPCHK(hipGetLastError());
  }

  void eam_table_eval(flyg_eam_s& E, int kind, int a, int b, double const* x, long m, int deriv, double* out) {
    int n = E.tab.ntypes;
    require(a >= 0 && a < n && b >= 0 && b < n, "type index out of range");
    require(deriv >= 0 && deriv <= 2, "deriv must be 0, 1 or 2");
    SplineDesc s = kind == 0 ? E.tab.F[a] : kind == 1 ? E.tab.phi[a + n * b] : E.tab.V[a > b ? a + n * b : b + n * a];
    DBuf<double> dx, dout;
    dx.reserve(m);
    dout.reserve(m);
    hipStream_t st = E.ctx->stream;
    HIPCHK(hipMemcpyAsync(dx.get(), x, m * sizeof(double), hipMemcpyHostToDevice, st));
    k_table_eval<<<static_cast<unsigned>((m + 255) / 256), 256, 0, st>>>(E.tab, s, dx.get(), m, deriv, dout.get(),
                                                                         E.ctx->dflags.get());
    HIPCHK(hipMemcpyAsync(out, dout.get(), m * sizeof(double), hipMemcpyDeviceToHost, st));
    throw_flags(E.ctx->take_flags());
  }

  namespace {
    // Names one upload of staged host types, unique in the process (lists cache per-slot species by it).
    long next_types_stamp() {
      static std::atomic<long> counter{0};
      return ++counter;
    }
  }  // namespace

  void stage_atoms(flyg_eam_s& E, uint32_t const* types, uint8_t const* frozen, long n, int where,
                   uint32_t const** d_types, uint8_t const** d_frozen) {
    if (!types && !frozen) {   // the handle's staged copy (stage_atoms_device or an earlier host call)
      require(E.staged_n == n, "no staged species and frozen flags for this many atoms");
      *d_types = E.types.get();
      *d_frozen = E.frozen.get();
      return;
    }
    require(types && frozen, "types and frozen must both be given or both be null");
    if (where == FLYG_DEVICE) {
      *d_types = types;
      *d_frozen = frozen;
      return;
    }
    bool same_t = static_cast<long>(E.last_types.size()) == n &&
                  std::memcmp(E.last_types.data(), types, n * sizeof(uint32_t)) == 0;
    bool same_f = static_cast<long>(E.last_frozen.size()) == n &&
                  std::memcmp(E.last_frozen.data(), frozen, n * sizeof(uint8_t)) == 0;
    int single = -1;
    if (!same_t) {   // validate before anything staged changes: a rejected call leaves no stale state
      single = n > 0 ? static_cast<int>(types[0]) : -1;
      for (long i = 0; i < n; ++i) {
        require(types[i] < static_cast<uint32_t>(E.tab.ntypes), "TypeID out of range");
        if (types[i] != types[0]) single = -1;
      }
    }
    // The device buffers may be reallocated below (contents lost): forget what they held first.
    if (!same_t || E.types.cap < static_cast<std::size_t>(n)) {
      E.last_types.clear();
      same_t = false;
    }
    if (!same_f || E.frozen.cap < static_cast<std::size_t>(n)) {
      E.last_frozen.clear();
      same_f = false;
    }
    E.types.reserve(n);
    E.frozen.reserve(n);
    if (!same_t) {
      HIPCHK(hipMemcpyAsync(E.types.get(), types, n * sizeof(uint32_t), hipMemcpyHostToDevice, E.ctx->stream));
      E.types_stamp = next_types_stamp();
      E.staged_single = single;
      E.last_types.assign(types, types + n);
    }
    if (!same_f) {
      HIPCHK(hipMemcpyAsync(E.frozen.get(), frozen, n * sizeof(uint8_t), hipMemcpyHostToDevice, E.ctx->stream));
      E.last_frozen.assign(frozen, frozen + n);
    }
    if (!same_t || !same_f) HIPCHK(hipStreamSynchronize(E.ctx->stream));
    E.staged_n = n;
    *d_types = E.types.get();
    *d_frozen = E.frozen.get();
  }

  void stage_atoms_device(flyg_eam_s& E, uint32_t const* types, uint8_t const* frozen, long n) {
    require(types && frozen, "null argument");
    E.staged_n = -1;
    E.last_types.clear();   // contents no longer match any host array
    E.last_frozen.clear();
    E.types.reserve(n);
    E.frozen.reserve(n);
    HIPCHK(hipMemcpyAsync(E.types.get(), types, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, E.ctx->stream));
    HIPCHK(hipMemcpyAsync(E.frozen.get(), frozen, n * sizeof(uint8_t), hipMemcpyDeviceToDevice, E.ctx->stream));
    E.types_stamp = next_types_stamp();
    E.staged_single = -1;   // not inspected on the host: the kernels treat the species as several
    E.staged_n = n;
  }

}  // namespace flyg
