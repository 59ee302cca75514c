// Neighbour-list build and update on gfx950 (replaces neigh::List, list.cpp:37-165).
//
// Rebuild pipeline (all on the device, one HIP stream):
//   1. k_entries: canonical real positions (List::rebuild copy-in, list.cpp:68-72) and their ghost images
//      (List::make_ghosts, list.cpp:100-132)
//   2. k_cell_count: the HyperGrid cell of each, counted with atomics whose return value is the entry's
//      place in arrival order
//   3. exclusive scan of the cell counts (which clears them for the next build)
//   4. scatter of the packed ids by cell, then each cell sorted by packed id, so the result does not
//      depend on the atomics
//   5. k_build_rows: every (real, image) of an atom's 27 cells with d^2 < r_cut^2 (strict,
//      list.cpp:146,159) goes to its row of an ELL table: n rows x K packed 32-bit entries, and to a second table
//      by slot (cell order): 16-bit indices into the tile's staged entries when the list is tiled, else packed entries
//      that name slots.
// Six launches and one synchronisation; the state the host needs is written to pinned memory.
// The distance tests, canonical images and ghost chains round exactly like the reference's FP64
// expressions (no FMA contraction), so the pair sets equal the reference's at rebuild time.
// Ghosts are not kept after the build: an entry stores (shift code, real index) and the pair kernels
// add the shift vector to the live real position, so update() touches only the N real atoms.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <numeric>

#include "eam_host.hpp"

namespace flyg {

  namespace {

    constexpr int TPB = 256;

    __device__ inline void canon_image(BoxDesc const& b, double* x) {
#pragma clang fp contract(off)
      if (b.ortho) {
        for (int k = 0; k < 3; ++k) x[k] = x[k] - b.ext[k] * floor(x[k] * b.inv_ext[k]);
        return;
      }
      double f[3];
      for (int r = 0; r < 3; ++r) f[r] = (b.Binv[r][0] * x[0] + b.Binv[r][1] * x[1]) + b.Binv[r][2] * x[2];
      for (int r = 0; r < 3; ++r) f[r] = f[r] - floor(f[r]);
      for (int r = 0; r < 3; ++r) x[r] = (b.B[r][0] * f[0] + b.B[r][1] * f[1]) + b.B[r][2] * f[2];
    }

    // OrthoGrid::gen_image (orthorhombic.hpp:54-74) / TriGrid::gen_image (triclinic.hpp:47-71).
    __device__ inline bool gen_image(BoxDesc const& b, double rc, int sign, double* x, int ax) {
#pragma clang fp contract(off)
      if (b.ortho) {
        if (sign > 0) {
          if (x[ax] < rc) {
            x[ax] += b.ext[ax];
            return true;
          }
        } else if (x[ax] > b.ext[ax] - rc) {
          x[ax] -= b.ext[ax];
          return true;
        }
        return false;
      }
      if (sign > 0) {
        double d = (x[0] * b.hyper[0][ax] + x[1] * b.hyper[1][ax]) + x[2] * b.hyper[2][ax];
        if (d < rc) {
          for (int r = 0; r < 3; ++r) x[r] = x[r] + b.B[r][ax];
          return true;
        }
      } else {
        double d = ((b.B[0][ax] - x[0]) * b.hyper[0][ax] + (b.B[1][ax] - x[1]) * b.hyper[1][ax])
                   + (b.B[2][ax] - x[2]) * b.hyper[2][ax];
        if (d < rc) {
          for (int r = 0; r < 3; ++r) x[r] = x[r] - b.B[r][ax];
          return true;
        }
      }
      return false;
    }

    // Position of the image with shift code s of a real atom at x: basis columns added axis by axis
    // (the chain make_ghosts produces).
    __device__ inline void image_of(BoxDesc const& b, unsigned s, double* x) {
#pragma clang fp contract(off)
      int sa[3] = {static_cast<int>(s % 3) - 1, static_cast<int>((s / 3) % 3) - 1, static_cast<int>(s / 9) - 1};
      for (int ax = 0; ax < 3; ++ax) {
        if (sa[ax] > 0) {
          for (int r = 0; r < 3; ++r) x[r] = x[r] + b.B[r][ax];
        } else if (sa[ax] < 0) {
          for (int r = 0; r < 3; ++r) x[r] = x[r] - b.B[r][ax];
        }
      }
    }

    // HyperGrid::cell_idx (hypergrid.hpp:74-99): clamp(int((x + cell) / cell)) per axis, x fastest.
    __device__ inline int cell_idx(GridDesc const& g, double const* x, int* c3) {
#pragma clang fp contract(off)
      int idx = 0;
      for (int k = 0; k < 3; ++k) {
        int i = static_cast<int>((x[k] + g.cell[k]) * g.inv_cell[k]);
        i = i < 0 ? 0 : (i > g.shape[k] - 1 ? g.shape[k] - 1 : i);
        c3[k] = i;
        idx += i * g.prod[k];
      }
      return idx;
    }

    __device__ inline double dist2(double const* a, double const* b) {
#pragma clang fp contract(off)
      double dx = a[0] - b[0], dy = a[1] - b[1], dz = a[2] - b[2];
      return (dx * dx + dy * dy) + dz * dz;
    }

    __global__ void k_update(double4* __restrict__ pos, double const* __restrict__ d, long n, int const* __restrict__ rank,
                             double4* __restrict__ gpos) {
      long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
      if (i >= n) return;
      double4 p = pos[i];
      p.x -= d[3 * i];
      p.y -= d[3 * i + 1];
      p.z -= d[3 * i + 2];
      pos[i] = p;
      double4* g = gpos + rank[i];   // its w slot may hold the atom's species: kept
      g->x = p.x;
      g->y = p.y;
      g->z = p.z;
    }

    __global__ void k_positions(double4 const* __restrict__ pos, long n, double* __restrict__ out) {
      long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
      if (i >= n) return;
      double4 p = pos[i];
      out[3 * i] = p.x;
      out[3 * i + 1] = p.y;
      out[3 * i + 2] = p.z;
    }

    // for_neighbours(i, r_cut) with the image chain: count, then write (j, shift, dr) rows.
    template <bool WRITE>
    __global__ void k_export(BoxDesc b, double rc, double4 const* __restrict__ pos, unsigned const* __restrict__ nbr,
                             int const* __restrict__ ncnt, int K, long n, long long const* __restrict__ off,
                             int* __restrict__ counts, int* __restrict__ oj, int* __restrict__ os, double* __restrict__ odr) {
      long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
      if (i >= n) return;
      double4 p = pos[i];
      double xi[3] = {p.x, p.y, p.z};
      int c = 0;
      long long o = WRITE ? off[i] : 0;
      int const cnt = min(ncnt[i], K);
      for (int k = 0; k < cnt; ++k) {
        unsigned e = nbr[i * static_cast<long>(K) + k];
        unsigned j = e & NB_IDX_MASK, s = e >> NB_SHIFT_BITS;
        double4 q = pos[j];
        double xn[3] = {q.x, q.y, q.z};
        image_of(b, s, xn);
        double dr[3], r2;
        {
#pragma clang fp contract(off)
          for (int r = 0; r < 3; ++r) dr[r] = xn[r] - xi[r];
          r2 = (dr[0] * dr[0] + dr[1] * dr[1]) + dr[2] * dr[2];
        }
        if (r2 < rc * rc) {
          if (WRITE) {
            oj[o + c] = static_cast<int>(j);
            os[o + c] = static_cast<int>(s);
            for (int r = 0; r < 3; ++r) odr[3 * (o + c) + r] = dr[r];
          }
          ++c;
        }
      }
      if (!WRITE) counts[i] = c;
    }

    // ---- single-sync rebuild path ----------------------------------------------------------------
    // lstate[0] ghosts generated, [1] longest row, [3] overflow bits, [4 + l] entries of the fullest tile of shape l,
    // [8 + l] tiles of shape l that hold atoms, [12] atoms sampled, [13] others that share their cells.
    enum : unsigned { OV_GHOST = 1u };

    // The tile shapes a build could take; workgroups [first[l], first[l + 1]) of k_rank_place look at shape l, those
    // after them place the entries.
    struct TileKinds {
      TileGrid g[TILE_KINDS];
      unsigned first[TILE_KINDS + 1];
    };

    // Slots for g images per thread, one atomic per workgroup of ETPB threads (prefix sums of the lanes' counts and
    // of the wavefronts' totals): the counter is one address, and an atomic per wavefront on it took 100 us
    // at a million atoms.  Slot order is free: the rank placement sorts every cell by packed id
    // afterwards.  Every thread of the workgroup must call it.
    constexpr int ETPB = 1024;

    __device__ inline unsigned ghost_slots(unsigned g, unsigned* st) {
      __shared__ unsigned wsum[ETPB / 64];
      __shared__ unsigned wbase;
      int const wl = static_cast<int>(threadIdx.x & 63), w = static_cast<int>(threadIdx.x >> 6);
      unsigned incl = g;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        unsigned t = __shfl_up(incl, o, 64);
        if (wl >= o) incl += t;
      }
      if (wl == 63) wsum[w] = incl;
      __syncthreads();
      if (threadIdx.x == 0) {
        unsigned total = 0;
        for (int q = 0; q < ETPB / 64; ++q) total += wsum[q];
        wbase = total > 0 ? atomicAdd(&st[0], total) : 0u;
      }
      __syncthreads();
      unsigned before = wbase;
      for (int q = 0; q < w; ++q) before += wsum[q];
      return before + (incl - g);
    }

    // The reference's chain of gen_image calls (any box): images of images, axis by axis.
    __device__ inline void ghosts_chain(BoxDesc const& b, GridDesc const& g, double const* x, bool inr, long i, long n,
                                        double4* __restrict__ ent, unsigned* __restrict__ eid, unsigned* __restrict__ st,
                                        long gcap) {
      double cx[27][3];
      int cs[27];
      int m = 1;
      cx[0][0] = x[0];
      cx[0][1] = x[1];
      cx[0][2] = x[2];
      cs[0] = 13;
      int const pow3[3] = {1, 3, 9};
      for (int ax = 0; ax < 3 && inr; ++ax) {
        if (!b.per[ax]) continue;
        int const end = m;
        for (int sgn = 1; sgn >= -1; sgn -= 2) {
          for (int c = 0; c < end; ++c) {
            double im[3] = {cx[c][0], cx[c][1], cx[c][2]};
            if (gen_image(b, g.rc, sgn, im, ax)) {
              cx[m][0] = im[0];
              cx[m][1] = im[1];
              cx[m][2] = im[2];
              cs[m] = cs[c] + sgn * pow3[ax];
              ++m;
            }
          }
        }
      }
      unsigned const ng = static_cast<unsigned>(m - 1);
      unsigned const base = ghost_slots(ng, st);
      for (int k = 1; k < m; ++k) {
        long const slot = static_cast<long>(base) + (k - 1);
        if (slot >= gcap) {
          atomicOr(&st[3], static_cast<unsigned>(OV_GHOST));
          return;
        }
        ent[n + slot] = make_double4(cx[k][0], cx[k][1], cx[k][2], 0.0);
        eid[n + slot] = (static_cast<unsigned>(cs[k]) << NB_SHIFT_BITS) | static_cast<unsigned>(i);
      }
    }

    // Reals and ghosts (capacity gcap; the counter keeps counting past it so the host can resize).  Launched with whole wavefronts.  Orthorhombic boxes: whether an axis contributes a
    // +1 / -1 image depends only on the atom's own coordinate on that axis, so the images are the product of the
    // per-axis choices (the same set, and the same coordinates, as the reference's chain) and live in
    // registers; other boxes follow the chain of gen_image calls.  One instantiation per box kind: the
    // chain's per-lane arrays live in scratch memory, which the orthorhombic form does not need.
    template <bool ORTHO>
    __global__ __launch_bounds__(ETPB) void k_entries(BoxDesc b, GridDesc g, double const* __restrict__ xyz, long n, double4* __restrict__ pos,
                              double4* __restrict__ ent, unsigned* __restrict__ eid, unsigned* __restrict__ st,
                              long gcap) {
      long const i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
      bool const inr = i < n;
      double x[3] = {0, 0, 0};
      if (inr) {
        x[0] = xyz[3 * i];
        x[1] = xyz[3 * i + 1];
        x[2] = xyz[3 * i + 2];
        canon_image(b, x);
        double4 const p = make_double4(x[0], x[1], x[2], 0.0);
        pos[i] = p;
        ent[i] = p;
        eid[i] = (13u << NB_SHIFT_BITS) | static_cast<unsigned>(i);
      }
      if constexpr (ORTHO) {
        bool up[3], dn[3];
        unsigned ng = inr ? 1 : 0;
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
          up[ax] = inr && b.per[ax] && x[ax] < g.rc;
          dn[ax] = inr && b.per[ax] && x[ax] > b.ext[ax] - g.rc;
          ng *= 1u + (up[ax] ? 1u : 0u) + (dn[ax] ? 1u : 0u);
        }
        ng = inr ? ng - 1u : 0u;
        unsigned const base = ghost_slots(ng, st);
        if (ng == 0) return;
        unsigned k = 0;
        for (int code = 0; code < 27; ++code) {
          int const s0 = code % 3 - 1, s1 = code / 3 % 3 - 1, s2 = code / 9 - 1;
          bool const use = (s0 == 0 || (s0 > 0 ? up[0] : dn[0])) && (s1 == 0 || (s1 > 0 ? up[1] : dn[1])) &&
                           (s2 == 0 || (s2 > 0 ? up[2] : dn[2]));
          if (code == 13 || !use) continue;
          long const slot = static_cast<long>(base) + k;
          ++k;
          if (slot >= gcap) {
            atomicOr(&st[3], static_cast<unsigned>(OV_GHOST));
            return;
          }
          double im[3] = {x[0], x[1], x[2]};
          {
#pragma clang fp contract(off)
            if (s0 > 0) im[0] += b.ext[0];
            if (s0 < 0) im[0] -= b.ext[0];
            if (s1 > 0) im[1] += b.ext[1];
            if (s1 < 0) im[1] -= b.ext[1];
            if (s2 > 0) im[2] += b.ext[2];
            if (s2 < 0) im[2] -= b.ext[2];
          }
          ent[n + slot] = make_double4(im[0], im[1], im[2], 0.0);
          eid[n + slot] = (static_cast<unsigned>(code) << NB_SHIFT_BITS) | static_cast<unsigned>(i);
        }
      } else {
        ghosts_chain(b, g, x, inr, i, n, ent, eid, st, gcap);
      }
    }

    __device__ inline long live_entries(unsigned const* st, long n, long gcap) {
      long g = static_cast<long>(st[0]);
      return n + (g < gcap ? g : gcap);
    }

    // Cell of every entry and its place in the cell in arrival order.  Counts: cnt[c] entries of cell c,
    // cnt[nc1 + c] real ones (one scan of both gives the cell starts and, less the first half's total, the
    // first slot of each cell's reals).  A launch of its own: inside k_entries a corner atom's 26 ghosts would wait
    // for one atomic's return after the other (28 us instead of 6 + 7 at 54.5k atoms).
    __global__ void k_cell_count(GridDesc g, double4 const* __restrict__ ent, long n, long gcap,
                                 unsigned const* __restrict__ st, int* __restrict__ ecell, int* __restrict__ earr,
                                 int* __restrict__ cnt, long nc1) {
      long e = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
      if (e >= live_entries(st, n, gcap)) return;
      double4 p = ent[e];
      double x[3] = {p.x, p.y, p.z};
      int c3[3];
      int c = cell_idx(g, x, c3);
      ecell[e] = c;
      if (e < n) atomicAdd(&cnt[nc1 + c], 1);
      earr[e] = atomicAdd(&cnt[c], 1);
    }

    // Counting-sort scatter of the packed ids only (order inside a cell follows the atomics).
    __global__ void k_scatter_ids(unsigned const* __restrict__ eid, int const* __restrict__ ecell,
                                  int const* __restrict__ earr, long n, long gcap, unsigned const* __restrict__ st,
                                  int const* __restrict__ cstart, unsigned* __restrict__ usid) {
      long e = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
      if (e >= live_entries(st, n, gcap)) return;
      usid[cstart[ecell[e]] + earr[e]] = eid[e];
    }

    // Places every entry at cell start + its rank among the cell's packed ids: cells come out sorted by
    // id whatever order the atomics took, so rows (and every sum over them) are reproducible.  A real
    // atom also gets its slot of the gradient layout: the reals in this sorted order (the cell's first
    // real slot + the reals of the cell with smaller ids), with its position by slot.
    __global__ void k_rank_place(double4 const* __restrict__ ent, unsigned const* __restrict__ eid,
                                 int const* __restrict__ ecell, long n, long gcap, unsigned const* __restrict__ st,
                                 int const* __restrict__ cstart, long nc1, unsigned const* __restrict__ usid,
                                 double4* __restrict__ spos, unsigned* __restrict__ sid, int* __restrict__ rslot,
                                 int* __restrict__ order, int* __restrict__ rank_of, double4* __restrict__ gpos,
                                 TileKinds tk, unsigned* __restrict__ seen, unsigned* __restrict__ sample) {
      if (blockIdx.x < tk.first[TILE_KINDS]) {   // four lanes a tile: the entries it stages, and whether it holds atoms
        int l = 0;
        while (blockIdx.x >= tk.first[l + 1]) ++l;
        TileGrid const& tg = tk.g[l];
        int const w = static_cast<int>((blockIdx.x - tk.first[l]) * blockDim.x + threadIdx.x), t = w >> 2;
        int sum = 0, own = 0;
        if (t < tg.ntiles) {
          int const tx = t % tg.nt[0], ty = t / tg.nt[0] % tg.nt[1], tz = t / (tg.nt[0] * tg.nt[1]);
#pragma unroll
          for (int y = 0; y < 4; ++y) {   // the lines of one z
            int hb, he, ob, oe;
            tg.line(true, tx, ty, tz, 4 * (w & 3) + y, hb, he);
            tg.line(false, tx, ty, tz, 4 * (w & 3) + y, ob, oe);
            sum += cstart[he] - cstart[hb];
            own += cstart[nc1 + oe] - cstart[nc1 + ob];
          }
        }
        for (int o = 1; o < 4; o <<= 1) {
          sum += __shfl_xor(sum, o, 64);
          own += __shfl_xor(own, o, 64);
        }
        // One pair of atomics a workgroup: they all go to one line, several nanoseconds each.
        __shared__ int s_sum, s_used;
        if (threadIdx.x == 0) s_sum = s_used = 0;
        __syncthreads();
        for (int o = 32; o > 2; o >>= 1) sum = max(sum, __shfl_xor(sum, o, 64));
        int const used = __popcll(__ballot(own > 0)) / 4;
        if ((threadIdx.x & 63) == 0) {
          atomicMax(&s_sum, sum);
          atomicAdd(&s_used, used);
        }
        __syncthreads();
        if (threadIdx.x == 0) {
          atomicMax(&seen[l], static_cast<unsigned>(s_sum));
          atomicAdd(&seen[4 + l], static_cast<unsigned>(s_used));
        }
        return;
      }
      long e = (blockIdx.x - tk.first[TILE_KINDS]) * static_cast<long>(blockDim.x) + threadIdx.x;
      if (e >= live_entries(st, n, gcap)) return;
      int c = ecell[e];
      unsigned id = eid[e];
      int b = cstart[c], end = cstart[c + 1];
      unsigned const block = blockIdx.x - tk.first[TILE_KINDS];
      if (block % 64 == 0 && (block + 1) * static_cast<long>(blockDim.x) <= n) {   // a sample of the atoms' surroundings
        int others = end - b - 1;
        for (int o = 32; o > 0; o >>= 1) others += __shfl_xor(others, o, 64);
        if ((threadIdx.x & 63) == 0) {
          atomicAdd(&sample[0], 64u);
          atomicAdd(&sample[1], static_cast<unsigned>(others));
        }
      }
      int rank = 0, reals_before = 0;
      for (int q = b; q < end; ++q) {
        unsigned const u = usid[q];
        bool const lt = u < id;
        rank += lt ? 1 : 0;
        reals_before += (lt && (u >> NB_SHIFT_BITS) == 13u) ? 1 : 0;
      }
      spos[b + rank] = ent[e];
      sid[b + rank] = id;
      if (e < n) {   // the first n entries are the reals, entry e = atom e
        rslot[e] = b + rank;
        int const slot = cstart[nc1 + c] - cstart[nc1] + reals_before;
        order[slot] = static_cast<int>(e);
        rank_of[e] = slot;
        gpos[slot] = ent[e];
      }
    }

    // List::build_neigh_list (list.cpp:134-165): a wavefront walks the 3x3x3 block of cells around A
    // consecutive slots (atoms in cell order) with the strict r < r_c test of the reference, z outermost, x
    // innermost, each cell in packed-id order.  The up-to-three x-neighbouring cells of a (y, z) line are
    // consecutive cells (x fastest), so their sorted atoms are one contiguous range: 9 ranges, whose ends the
    // first nine lanes fetch at once.  A range holds 36 to 60 candidates in a metal at these cut-offs, one
    // coalesced chunk of 64; the chunks of three ranges are loaded before the first is tested, and hits are
    // taken in candidate order (ballot + prefix count), so a row is the sequence a single thread would produce.
    // A chunk yields about eight hits: they wait in a ring in LDS until 64 of them leave as one coalesced store.
    // Slots of one cell share the candidates' loads; a wavefront whose slots straddle cells walks each
    // cell's block in turn.
    // Small systems are bound by the chain of loads (A = 1: every atom a wavefront), large ones by the
    // candidates' L1 lookups (A = 4 loads them a quarter as often); BUILD_WIDE is where the two cross.
    //
    // Each row is written twice: by atom with atom indices (nbr), and by slot, in a tiled list with indices into the
    // tile's stage (the candidate's place in the tile's halo: the lines' entries one after the other), otherwise with
    // slots.  hst (pinned): the build counters, but [1] set when a row overflowed.
    constexpr long BUILD_WIDE = 24000;
    // Atoms a cell below which eight lanes an atom are faster than four atoms a wavefront.  Rebuild, us, by the two:
    // 26k atoms at 1, 4, 6, 8 atoms a cell 63.6/80.1, 59.1/68.5, 61.4/66.8, 66.0/65.1; 1M at 0.3 and 2 533/1095, 579/985.
    constexpr double SPARSE = 6.0;

    template <int A, bool TILED>
    __global__ __launch_bounds__(TPB) void k_build_rows(GridDesc g, double4 const* __restrict__ spos,
                                                        unsigned const* __restrict__ sid, int const* __restrict__ cstart,
                                                        int const* __restrict__ rslot, long n, unsigned* __restrict__ nbr,
                                                        int* __restrict__ ncnt, int K, unsigned* __restrict__ st,
                                                        int const* __restrict__ order, int const* __restrict__ rank_of,
                                                        TileGrid tg, unsigned* __restrict__ sslot, long live_cap,
                                                        unsigned* __restrict__ rows, int rowK, int* __restrict__ gcnt,
                                                        unsigned* __restrict__ hst) {
      if (blockIdx.x == 0 && threadIdx.x < LIST_STATE && threadIdx.x != 1) hst[threadIdx.x] = st[threadIdx.x];
      if constexpr (TILED) {
        long const live = live_entries(st, n, live_cap);
        for (long s = blockIdx.x * static_cast<long>(TPB) + threadIdx.x; s < live; s += static_cast<long>(gridDim.x) * TPB) {
          unsigned const en = sid[s];
          sslot[s] = (en & ~NB_IDX_MASK) | static_cast<unsigned>(rank_of[en & NB_IDX_MASK]);
        }
      }
      int const lane = static_cast<int>(threadIdx.x & 63);
      int const wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
      long const slot0 = (xcd_block(blockIdx.x, gridDim.x) * static_cast<long>(TPB / 64) + wave) * A;
      if (slot0 >= n) return;   // whole wavefronts leave together
      int const na = static_cast<int>(min(static_cast<long>(A), n - slot0));
      __shared__ unsigned ring[TPB / 64][A][128];
      __shared__ unsigned short ring16[TILED ? TPB / 64 : 1][A][128];
      double const rc2 = g.rc * g.rc;
      int atom[A], self[A], cell[A], cx[A], cy[A], cz[A], cnt[A];
      double xi[A][3];
#pragma unroll
      for (int a = 0; a < A; ++a) {
        atom[a] = order[slot0 + min(a, na - 1)];
        self[a] = rslot[atom[a]];
      }
#pragma unroll
      for (int a = 0; a < A; ++a) {
        double4 const p = spos[self[a]];
        xi[a][0] = p.x;
        xi[a][1] = p.y;
        xi[a][2] = p.z;
        int c3[3];
        cell[a] = cell_idx(g, xi[a], c3);
        cx[a] = c3[0];
        cy[a] = c3[1];
        cz[a] = c3[2];
        cnt[a] = 0;
      }
      // Entries [k0, k0 + 64) of slot a's row, those below `c` (a wavefront runs in lockstep: its LDS accesses
      // need no barrier, only their program order).
      auto flush = [&](int a, int k0, int c) {
        int const k = k0 + lane;
        __builtin_amdgcn_wave_barrier();
        if (k < c && k < K) {
          unsigned const en = ring[wave][a][k & 127];
          nbr[atom[a] * static_cast<long>(K) + k] = en;
          if constexpr (!TILED)
            rows[(slot0 + a) * rowK + k] = (en & ~NB_IDX_MASK) | static_cast<unsigned>(rank_of[en & NB_IDX_MASK]);
        }
        if constexpr (TILED) {   // two blocks of 32 entries, two entries a lane
          int const k2 = k0 + (lane >> 4) * 32 + (lane & 15);
          if (lane < 32 && k2 < c && k2 < K) {
            unsigned const w = ring16[wave][a][k2 & 127] | (static_cast<unsigned>(ring16[wave][a][(k2 + 16) & 127]) << 16);
            rows[((slot0 + a) * rowK + k0) / 2 + lane] = w;
          }
        }
        __builtin_amdgcn_wave_barrier();
      };
      int done = 0;   // slots whose rows are written
      while (done < na) {
        int c0 = cell[0], x = cx[0], y0 = cy[0], z0 = cz[0];
#pragma unroll
        for (int a = 1; a < A; ++a)
          if (a == done) {
            c0 = cell[a];
            x = cx[a];
            y0 = cy[a];
            z0 = cz[a];
          }
        int rb = 0, re = 0;   // lane l < 9: range l
        int loc = 0;          // ... and what turns a place in the sorted entries into one in the tile's stage
        if constexpr (TILED) {
          int const tx = tg.of(0, x), ty = tg.of(1, y0), tz = tg.of(2, z0);
          int const q = lane & 15;
          int cb, ce;
          tg.line(true, tx, ty, tz, q, cb, ce);
          int const lb = cstart[cb], len = cstart[ce] - lb;
          int incl = len;
#pragma unroll
          for (int o = 1; o < 16; o <<= 1) {
            int const t = __shfl_up(incl, o, 16);
            if (q >= o) incl += t;
          }
          int const shift = (incl - len) - lb;   // by line of the tile
          int const ly = y0 - 1 + lane % 3 - tg.halo_lo(1, ty), lz = z0 - 1 + lane / 3 - tg.halo_lo(2, tz);
          loc = __shfl(shift, (ly + 4 * lz) & 15, 64);   // of a line outside the grid: not used
        }
        if (lane < 9) {
          int const y = y0 - 1 + lane % 3, z = z0 - 1 + lane / 3;
          if (y >= 0 && y < g.shape[1] && z >= 0 && z < g.shape[2]) {
            int const line = y * g.prod[1] + z * g.prod[2];
            rb = cstart[max(x - 1, 0) * g.prod[0] + line];
            re = cstart[min(x + 1, g.shape[0] - 1) * g.prod[0] + line + 1];
          }
        }
        auto test = [&](double4 const& q, unsigned en, int s, int shift) {
          double const xn[3] = {q.x, q.y, q.z};   // far away on lanes without a candidate
#pragma unroll
          for (int a = 0; a < A; ++a) {
            if (a >= na || cell[a] != c0) continue;
            bool const hit = s != self[a] && dist2(xi[a], xn) < rc2;
            unsigned long long const m = __ballot(hit);
            int const before = __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(m >> 32),
                                                         __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(m), 0u));
            if (hit) {
              ring[wave][a][(cnt[a] + before) & 127] = en;
              if constexpr (TILED) ring16[wave][a][(cnt[a] + before) & 127] = static_cast<unsigned short>(s + shift);
            }
            int const c = cnt[a] + __popcll(m);
            if ((c ^ cnt[a]) & ~63) flush(a, cnt[a] & ~63, c & ~63);   // a block of 64 is full
            cnt[a] = c;
          }
        };
        for (int z = 0; z < 3; ++z) {
          int b[3], e[3], sh[3];
          double4 q[3];
          unsigned en[3];
#pragma unroll
          for (int u = 0; u < 3; ++u) {
            b[u] = __builtin_amdgcn_readlane(rb, 3 * z + u);
            e[u] = __builtin_amdgcn_readlane(re, 3 * z + u);
            sh[u] = TILED ? __builtin_amdgcn_readlane(loc, 3 * z + u) : 0;
            int const s = b[u] + lane;
            en[u] = 0;
            q[u] = make_double4(1e200, 0.0, 0.0, 0.0);
            if (s < e[u]) {
              q[u] = spos[s];
              en[u] = sid[s];
            }
          }
#pragma unroll
          for (int u = 0; u < 3; ++u) {
            test(q[u], en[u], b[u] + lane, sh[u]);
            for (int s0 = b[u] + 64; s0 < e[u]; s0 += 64) {   // the rest of a long range
              int const s = s0 + lane;
              double4 c = make_double4(1e200, 0.0, 0.0, 0.0);
              unsigned id = 0;
              if (s < e[u]) {
                c = spos[s];
                id = sid[s];
              }
              test(c, id, s, sh[u]);
            }
          }
        }
        int next = na;   // the first later slot of another cell (slots are in cell order)
#pragma unroll
        for (int a = A - 1; a > 0; --a)
          if (a > done && a < na && cell[a] != c0) next = a;
        done = next;
      }
#pragma unroll
      for (int a = 0; a < A; ++a)
        if (a < na) flush(a, cnt[a] & ~63, cnt[a]);
      if (lane < A && lane < na) {
        int c = cnt[0], i = atom[0];
#pragma unroll
        for (int a = 1; a < A; ++a)
          if (a == lane) {
            c = cnt[a];
            i = atom[a];
          }
        ncnt[i] = c;
        gcnt[slot0 + lane] = c;
        // Only overflowing rows report their length (the host widens the rows to the longest one): an
        // atomic per atom on the one counter serialised the kernel (half of its time).
        if (c > K) {
          atomicMax(&st[1], static_cast<unsigned>(c));
          hst[1] = 1u;
        }
      }
    }

    // The same for a dilute system, whose ranges hold a few candidates each: eight lanes an atom, so a wavefront walks the
    // blocks of eight atoms at once instead of a mostly empty chunk of 64 after the other.  Lists of plain rows only.
    constexpr int SPARSE_LANES = 8;
    constexpr int SPARSE_UNROLL = 4;   // chunks of candidates loaded before the first is tested

    __global__ __launch_bounds__(TPB) void k_build_rows_sparse(GridDesc g, double4 const* __restrict__ spos,
                                                               unsigned const* __restrict__ sid,
                                                               int const* __restrict__ cstart, int const* __restrict__ rslot,
                                                               long n, unsigned* __restrict__ nbr, int* __restrict__ ncnt,
                                                               int K, unsigned* __restrict__ st,
                                                               int const* __restrict__ order, int const* __restrict__ rank_of,
                                                               unsigned* __restrict__ rows, int* __restrict__ gcnt,
                                                               unsigned* __restrict__ hst) {
      if (blockIdx.x == 0 && threadIdx.x < LIST_STATE && threadIdx.x != 1) hst[threadIdx.x] = st[threadIdx.x];
      constexpr int L = SPARSE_LANES, U = SPARSE_UNROLL;
      long const gid = xcd_block(blockIdx.x, gridDim.x) * static_cast<long>(TPB) + threadIdx.x, slot = gid / L;
      int const lane = static_cast<int>(gid % L), gbase = static_cast<int>(threadIdx.x & 63) - lane;
      if (slot >= n) return;   // whole groups leave together
      int const atom = order[slot], self = rslot[atom];
      double4 const p = spos[self];
      double const xi[3] = {p.x, p.y, p.z}, rc2 = g.rc * g.rc;
      int c3[3];
      cell_idx(g, xi, c3);
      int cnt = 0;
      unsigned* row = nbr + atom * static_cast<long>(K);
      unsigned* srow = rows + slot * K;
      int const x0 = max(c3[0] - 1, 0), x1 = min(c3[0] + 2, g.shape[0]);
      for (int z = max(c3[2] - 1, 0); z < min(c3[2] + 2, g.shape[2]); ++z)
        for (int y = max(c3[1] - 1, 0); y < min(c3[1] + 2, g.shape[1]); ++y) {
          int const line = y * g.prod[1] + z * g.prod[2];
          int const b = cstart[x0 * g.prod[0] + line], end = cstart[(x1 - 1) * g.prod[0] + line + 1];
          for (int s0 = b; s0 < end; s0 += U * L) {
            bool hit[U];
            unsigned en[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
              int const s = s0 + u * L + lane;
              hit[u] = false;
              en[u] = 0;
              if (s < end && s != self) {
                double4 const q = spos[s];
                en[u] = sid[s];
                double const xn[3] = {q.x, q.y, q.z};
                hit[u] = dist2(xi, xn) < rc2;
              }
            }
            int rk[U];
#pragma unroll
            for (int u = 0; u < U; ++u) rk[u] = hit[u] ? rank_of[en[u] & NB_IDX_MASK] : 0;
#pragma unroll
            for (int u = 0; u < U; ++u) {
              unsigned long long const m = __ballot(hit[u]);
              unsigned const gm = static_cast<unsigned>((m >> gbase) & ((1ull << L) - 1ull));
              int const k = cnt + __popc(gm & ((1u << lane) - 1u));
              if (hit[u] && k < K) {
                row[k] = en[u];
                srow[k] = (en[u] & ~NB_IDX_MASK) | static_cast<unsigned>(rk[u]);
              }
              cnt += __popc(gm);
            }
          }
        }
      if (lane == 0) {
        ncnt[atom] = cnt;
        gcnt[slot] = cnt;
        if (cnt > K) {
          atomicMax(&st[1], static_cast<unsigned>(cnt));
          hst[1] = 1u;
        }
      }
    }

    constexpr int SCAN_B = 1024;

    // First level of an exclusive scan of src into dst (which may be src); clear: src is zeroed, and so are
    // the LIST_STATE words at cst.
    __global__ void k_scan_block(int* src, int* dst, int n, int* __restrict__ sums, bool clear, unsigned* cst) {
      __shared__ int wsum[SCAN_B / 64];
      int gi = blockIdx.x * SCAN_B + threadIdx.x;
      int v = gi < n ? src[gi] : 0;
      if (clear) {
        if (gi < n) src[gi] = 0;
        if (gi < LIST_STATE) cst[gi] = 0u;
      }
      int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
      int inc = v;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        int t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
      }
      if (lane == 63) wsum[w] = inc;
      __syncthreads();
      if (w == 0) {
        int s = lane < SCAN_B / 64 ? wsum[lane] : 0;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          int t = __shfl_up(s, o, 64);
          if (lane >= o) s += t;
        }
        if (lane < SCAN_B / 64) wsum[lane] = s;
      }
      __syncthreads();
      int before = (w > 0 ? wsum[w - 1] : 0) + inc - v;
      if (gi < n) dst[gi] = before;
      if (threadIdx.x == SCAN_B - 1) sums[blockIdx.x] = wsum[SCAN_B / 64 - 1];
    }

    // Exclusive scan of up to SCAN_B * SCAN_RUN values in one workgroup: thread t owns a run of `per`
    // consecutive values (a multiple of four, kept in registers), the runs' totals are scanned across the block.
    // Both arrays hold scan_room(n) values and are 16-byte aligned: a run is read and written four values at a time.
    constexpr int SCAN_RUN = 16;

    __global__ __launch_bounds__(SCAN_B) void k_scan_one(int* src, int* dst, int n, bool clear, unsigned* cst) {
      __shared__ int wsum[SCAN_B / 64];
      int const per = ((n + SCAN_B - 1) / SCAN_B + 3) & ~3;
      int const b = static_cast<int>(threadIdx.x) * per;
      int val[SCAN_RUN];
      int v = 0;
#pragma unroll
      for (int q = 0; q < SCAN_RUN; q += 4) {
        int4 t = make_int4(0, 0, 0, 0);
        if (q < per && b + q < n) t = *reinterpret_cast<int4 const*>(src + b + q);
        val[q] = t.x;
        val[q + 1] = b + q + 1 < n ? t.y : 0;
        val[q + 2] = b + q + 2 < n ? t.z : 0;
        val[q + 3] = b + q + 3 < n ? t.w : 0;
        v += val[q] + val[q + 1] + val[q + 2] + val[q + 3];
      }
      if (clear) {
#pragma unroll
        for (int q = 0; q < SCAN_RUN; q += 4)
          if (q < per && b + q < n) *reinterpret_cast<int4*>(src + b + q) = make_int4(0, 0, 0, 0);
        if (threadIdx.x < LIST_STATE) cst[threadIdx.x] = 0u;
      }
      int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
      int inc = v;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        int t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
      }
      if (lane == 63) wsum[w] = inc;
      __syncthreads();
      if (w == 0) {
        int s = lane < SCAN_B / 64 ? wsum[lane] : 0;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          int t = __shfl_up(s, o, 64);
          if (lane >= o) s += t;
        }
        if (lane < SCAN_B / 64) wsum[lane] = s;
      }
      __syncthreads();
      int run = (w > 0 ? wsum[w - 1] : 0) + inc - v;
#pragma unroll
      for (int q = 0; q < SCAN_RUN; q += 4) {
        int4 t;
        t.x = run;
        t.y = t.x + val[q];
        t.z = t.y + val[q + 1];
        t.w = t.z + val[q + 2];
        run = t.w + val[q + 3];
        if (q < per && b + q < n) *reinterpret_cast<int4*>(dst + b + q) = t;
      }
    }

    __global__ void k_scan_add(int* __restrict__ data, int n, int const* __restrict__ sums) {
      int gi = blockIdx.x * SCAN_B + threadIdx.x;
      if (gi < n) data[gi] += sums[blockIdx.x];
    }

    inline unsigned nblk(long n, int t) { return static_cast<unsigned>((n + t - 1) / t); }

  }  // namespace

  void exclusive_scan(flyg_ctx_s& ctx, int* src, int* dst, int n, DBuf<int>& tmp, unsigned* clear_state) {
    if (n <= 0) return;
    bool const clear = clear_state != nullptr;
    if (n <= SCAN_B * SCAN_RUN) {   // one launch: each launch in a stream costs several microseconds
      k_scan_one<<<1, SCAN_B, 0, ctx.stream>>>(src, dst, n, clear, clear_state);
      HIPCHK(hipGetLastError());
      return;
    }
    int nb = static_cast<int>((n + SCAN_B - 1) / SCAN_B);
    // Workspace layout: [sums of this level | workspace of the next level]
    std::vector<int> offs;
    std::vector<int> sizes;
    int total = 0, cur = nb;
    while (true) {
      offs.push_back(total);
      sizes.push_back(cur);
      total += cur;
      if (cur <= 1) break;
      cur = (cur + SCAN_B - 1) / SCAN_B;
    }
    tmp.reserve(static_cast<std::size_t>(total) + 1);
    // Down-sweep of block sums.
    int* level_data = dst;
    int level_n = n;
    for (std::size_t l = 0; l < offs.size(); ++l) {
      int blocks = (level_n + SCAN_B - 1) / SCAN_B;
      k_scan_block<<<blocks, SCAN_B, 0, ctx.stream>>>(l == 0 ? src : level_data, level_data, level_n, tmp.get() + offs[l],
                                                     clear && l == 0, clear_state);
      if (blocks == 1) break;
      level_data = tmp.get() + offs[l];
      level_n = blocks;
    }
    // Up-sweep: add scanned block sums back, deepest level first.
    for (std::size_t l = offs.size(); l-- > 0;) {
      int ln = l == 0 ? n : sizes[l - 1];
      int* ld = l == 0 ? dst : tmp.get() + offs[l - 1];
      int blocks = (ln + SCAN_B - 1) / SCAN_B;
      if (blocks == 1) continue;
      k_scan_add<<<blocks, SCAN_B, 0, ctx.stream>>>(ld, ln, tmp.get() + offs[l]);
    }
    HIPCHK(hipGetLastError());
  }

  void shift_table(BoxDesc const& b, double3* out) {
    for (int s = 0; s < 27; ++s) {
      int sa[3] = {s % 3 - 1, (s / 3) % 3 - 1, s / 9 - 1};
      double v[3] = {0, 0, 0};
      for (int ax = 0; ax < 3; ++ax)
        for (int r = 0; r < 3; ++r) v[r] += sa[ax] * b.B[r][ax];
      out[s] = make_double3(v[0], v[1], v[2]);
    }
  }

  namespace {
    // Tile shapes (cells), largest first.  A larger tile stages fewer entries per atom (8, 12, 18 of them) but there are
    // fewer workgroups, each walking more rows.  Which is best depends on how the tiles fill the chip: three
    // workgroups of 512 threads run on each of 256 CUs, so 1000 tiles take little less than 1500 would.  Gradient,
    // us, one species, list cut-off 5.9 A, mixed / FP64, by 2x2x2 (tiles) / 1x2x2 / 1x1x2 / plain rows in slot order:
    //   27.6k atoms  42.5/51.6 (216)   31.3/39.8 (396)   24.4/33.4 (726)   21.8/30.0
    //   43.9k        48.7/64.2 (343)   36.2/49.6 (637)   39.2/53.0 (1183)  33.0/43.4
    //   54.0k        47.6/63.1 (343)   36.9/50.4 (686)   40.5/54.5 (1372)  38.2/50.5
    //   110k         64.0/93.4 (729)   69.9/97.6 (1458)  73.7/101 (2916)   81.7/111
    //   128k         102/151 (1000)    81.8/119 (1900)   92.0/124 (3610)   92.8/128
    //   686k         348/505 (4913)    346/501 (9537)    415/560 (18513)   581/815
    constexpr int TILE_SHAPES[TILE_KINDS][3] = {{2, 2, 2}, {1, 2, 2}, {1, 1, 2}};
    constexpr long TILE_ATOMS = 27000;      // fewer: plain rows are faster or equal in the passes together
    constexpr long TILE_LEAST = 600;        // a little over two for each CU
    // Atoms a cell below which a tile's rows are too few and too short.  512k atoms at 4, 6, 8, 11 a cell (metals have 13
    // and more), mixed gradient, us, by tiles / by rows: 217/103, 180/133, 172/181, 188/216.
    constexpr long TILE_CELL = 8;
    constexpr double TILE_SLOTS = 768.0;    // workgroups resident at once

    TileGrid tile_grid(GridDesc const& g, int level) {
      TileGrid t{};
      t.ntiles = 1;
      for (int k = 0; k < 3; ++k) {
        t.d[k] = TILE_SHAPES[level][k];
        t.shape[k] = g.shape[k];
        t.prod[k] = g.prod[k];
        t.nt[k] = std::max(1, (g.shape[k] - 2 + t.d[k] - 1) / t.d[k]);
        t.ntiles *= t.nt[k];
      }
      t.nc1 = g.ncells + 1l;
      return t;
    }

    // What an atom costs in tiles of a shape, in the cost of full tiles of 2x2x2 that fill every round of workgroups:
    // the shape's own factor, a stage so large that a CU holds fewer workgroups (40 KB for four of a gradient's
    // and two of an HVP's, 54 KB for three), the last round's idle slots at half their time (its workgroups have more of a CU to
    // themselves), and cells that the last tile of an axis lacks.
    double tile_cost(TileGrid const& t, int level, double used, double staged) {
      constexpr double factor[TILE_KINDS] = {1.0, 1.12, 1.3};
      double const rounds = used / TILE_SLOTS;
      double inner = 1, most = t.ntiles;
      for (int k = 0; k < 3; ++k) {
        inner *= t.shape[k] - 2;
        most *= t.d[k];
      }
      double const large = staged > 1530 ? 1.5 : (staged > 1100 ? 1.1 : 1.0);
      return factor[level] * large * (0.5 + 0.5 * std::ceil(rounds) / rounds) * (most / inner);
    }

    // The tile shape for a build, or -1: plain rows.  The largest shape that leaves TILE_LEAST tiles, if no other is
    // clearly cheaper.  seen: from what the build before counted, the tiles that hold atoms and the fullest one.
    // A first build takes the box to be filled evenly, and is done again if its own counts say otherwise (a particle
    // in vacuum leaves most tiles empty and the chip idle: 16k atoms in eight times their volume took 74 us a
    // gradient by tiles, 25 by rows).
    int choose_tiles(flyg_list_s const& nl, long n, bool seen, double* cost = nullptr) {
      if (n < TILE_ATOMS) return -1;
      GridDesc const& g = nl.grid;
      double const inner = static_cast<double>(g.shape[0] - 2) * (g.shape[1] - 2) * (g.shape[2] - 2);
      int best = -1;
      bool first = true;
      double least = 2.0;   // dearer than plain rows
      for (int level = 0; level < TILE_KINDS; ++level) {
        TileGrid const t = tile_grid(g, level);
        double const staged = n / inner * (t.d[0] + 2) * (t.d[1] + 2) * (t.d[2] + 2);
        bool const full = staged > 0.9 * TILE_MOST || (seen && nl.tile_full[level] > TILE_MOST);
        long const used = seen ? static_cast<long>(nl.tile_used[level]) : t.ntiles;
        if (full || used == 0 || n < TILE_CELL * t.d[0] * t.d[1] * t.d[2] * used) continue;
        double const c = tile_cost(t, level, static_cast<double>(used), staged);
        double const compared = first && used >= TILE_LEAST ? 0.93 * c : c;
        if (used >= TILE_LEAST) first = false;
        if (compared < least) {
          least = compared;
          best = level;
          if (cost) *cost = c;
        }
      }
      return best;
    }

    // Neighbours within the list's cut-off in a box filled evenly.
    double mean_row(flyg_list_s const& nl, long n) {
      double const vol = std::fabs(nl.box.B[0][0] * (nl.box.B[1][1] * nl.box.B[2][2] - nl.box.B[1][2] * nl.box.B[2][1]) -
                                   nl.box.B[0][1] * (nl.box.B[1][0] * nl.box.B[2][2] - nl.box.B[1][2] * nl.box.B[2][0]) +
                                   nl.box.B[0][2] * (nl.box.B[1][0] * nl.box.B[2][1] - nl.box.B[1][1] * nl.box.B[2][0]));
      return static_cast<double>(n) / vol * 4.18879 * nl.rc * nl.rc * nl.rc;
    }
  }  // namespace

  // One rebuild costs one host synchronisation: capacities (ghost slots, row length) come from the
  // previous build; the device records what it needed and the build is redone only on overflow.
  void list_rebuild(flyg_list_s& nl, double const* d_xyz, long n) {
    require(n > 0, "List::rebuild with no atoms");
    require(n < MAX_ATOMS, "too many atoms for the packed neighbour format");
    flyg_ctx_s& ctx = *nl.ctx;
    hipStream_t st = ctx.stream;
    if (!nl.hstate) HIPCHK(hipHostMalloc(reinterpret_cast<void**>(&nl.hstate), LIST_STATE * sizeof(unsigned), hipHostMallocDefault));
    nl.built = false;
    if (n != nl.n) {
      nl.gcap = 0;
      nl.K = 0;
    }
    if (n != nl.n || !std::equal(nl.tile_shape, nl.tile_shape + 3, nl.grid.shape)) nl.tile_seen = false;
    std::copy(nl.grid.shape, nl.grid.shape + 3, nl.tile_shape);
    nl.n = n;
    if (nl.gcap == 0) nl.gcap = std::max(4096l, n);
    if (nl.K == 0) {
      // Room for the rows of a uniform system and a fifth more: a first guess of 64 built most lists twice.
      nl.K = std::max(64, (static_cast<int>(std::min(1.2 * mean_row(nl, n), 512.0)) + 15) / 16 * 16);
    }
    int const nc = nl.grid.ncells;
    long const nc1 = nc + 1;
    nl.lstate.reserve(2 * LIST_STATE);
    nl.ccount.reserve(scan_room(2 * nc1));
    nl.cstart.reserve(scan_room(2 * nc1));   // cell starts, then the first real slot of each cell (offset)
    nl.pos.reserve(n);
    nl.ncnt.reserve(n);
    nl.rslot.reserve(n);
    nl.order.reserve(n);
    nl.rank.reserve(n);
    nl.gpos.reserve(n);
    nl.gcnt.reserve(n);
    if (nl.clear_cells != nc1) {   // a first build, another grid, or a build that ended in an error half way
      HIPCHK(hipMemsetAsync(nl.ccount.get(), 0, scan_room(2 * nc1) * sizeof(int), st));
      HIPCHK(hipMemsetAsync(nl.lstate.get(), 0, 2 * LIST_STATE * sizeof(unsigned), st));
    }
    nl.clear_cells = -1;

    TileKinds tk{};
    for (int l = 0; l < TILE_KINDS; ++l) tk.g[l] = tile_grid(nl.grid, l);
    for (int attempt = 0; attempt < 6; ++attempt) {
      // Two sets of state words in turn: the scan clears the other build's.
      unsigned* dst = nl.lstate.get() + LIST_STATE * nl.parity;
      unsigned* other = nl.lstate.get() + LIST_STATE * (1 - nl.parity);
      nl.parity = 1 - nl.parity;
      long const cap = n + nl.gcap;
      nl.ent.reserve(cap);
      nl.eid.reserve(cap);
      nl.ecell.reserve(cap);
      nl.earr.reserve(cap);
      nl.spos.reserve(cap);
      nl.sid.reserve(cap);
      nl.usid.reserve(cap);
      nl.nbr.reserve(static_cast<std::size_t>(n) * nl.K);
      double cost = 0;
      int const level = choose_tiles(nl, n, nl.tile_seen, &cost);
      nl.tiled = level >= 0;
      // The shape in use is looked at in every build, the others (not those with more tiles than a quarter of the
      // atoms) only while an even filling and what was seen disagree: three shapes take 5 us more at 54k atoms.
      bool const all = n >= TILE_ATOMS && (!nl.tile_seen || attempt > 0 || level != choose_tiles(nl, n, false));
      for (int l = 0; l < TILE_KINDS; ++l) {
        bool const look = l == level || (all && n >= 4l * tk.g[l].ntiles);
        tk.first[l + 1] = tk.first[l] + (look ? nblk(4l * tk.g[l].ntiles, TPB) : 0);
      }
      TileGrid const tg = nl.tiled ? tk.g[level] : TileGrid{};
      nl.rowK = nl.tiled ? (nl.K + 31) / 32 * 32 : nl.K;
      if (nl.tiled) nl.sslot.reserve(cap);
      nl.rows.reserve(static_cast<std::size_t>(n) * nl.rowK / (nl.tiled ? 2 : 1));
      nl.hstate[1] = 0;
      if (nl.box.ortho) {
        k_entries<true><<<nblk(n, ETPB), ETPB, 0, st>>>(nl.box, nl.grid, d_xyz, n, nl.pos.get(), nl.ent.get(),
                                                        nl.eid.get(), dst, nl.gcap);
      } else {
        k_entries<false><<<nblk(n, ETPB), ETPB, 0, st>>>(nl.box, nl.grid, d_xyz, n, nl.pos.get(), nl.ent.get(),
                                                        nl.eid.get(), dst, nl.gcap);
      }
      k_cell_count<<<nblk(cap, TPB), TPB, 0, st>>>(nl.grid, nl.ent.get(), n, nl.gcap, dst, nl.ecell.get(), nl.earr.get(),
                                                   nl.ccount.get(), nc1);
      exclusive_scan(ctx, nl.ccount.get(), nl.cstart.get(), static_cast<int>(2 * nc1), nl.scan_tmp, other);
      k_scatter_ids<<<nblk(cap, TPB), TPB, 0, st>>>(nl.eid.get(), nl.ecell.get(), nl.earr.get(), n, nl.gcap, dst,
                                                    nl.cstart.get(), nl.usid.get());
      k_rank_place<<<tk.first[TILE_KINDS] + nblk(cap, TPB), TPB, 0, st>>>(
          nl.ent.get(), nl.eid.get(), nl.ecell.get(), n, nl.gcap, dst, nl.cstart.get(), nc1, nl.usid.get(), nl.spos.get(),
          nl.sid.get(), nl.rslot.get(), nl.order.get(), nl.rank.get(), nl.gpos.get(), tk, dst + 4,
          dst + 12);
      auto rows = [&](auto k, int A) {
        k<<<nblk(n, A * (TPB / 64)), TPB, 0, st>>>(nl.grid, nl.spos.get(), nl.sid.get(), nl.cstart.get(), nl.rslot.get(), n,
                                                   nl.nbr.get(), nl.ncnt.get(), nl.K, dst, nl.order.get(), nl.rank.get(),
                                                   tg, nl.sslot.get(), nl.gcap, nl.rows.get(), nl.rowK, nl.gcnt.get(),
                                                   nl.hstate);
      };
      static_assert(TILE_ATOMS >= BUILD_WIDE, "a tiled list has enough atoms for four a wavefront");
      if (nl.tiled) {
        rows(k_build_rows<4, true>, 4);
      } else if (n >= BUILD_WIDE &&
                 n < SPARSE * (nl.grid.shape[0] - 2) * (nl.grid.shape[1] - 2) * (nl.grid.shape[2] - 2)) {
        k_build_rows_sparse<<<nblk(n, TPB / SPARSE_LANES), TPB, 0, st>>>(
            nl.grid, nl.spos.get(), nl.sid.get(), nl.cstart.get(), nl.rslot.get(), n, nl.nbr.get(), nl.ncnt.get(), nl.K, dst,
            nl.order.get(), nl.rank.get(), nl.rows.get(), nl.gcnt.get(), nl.hstate);
      } else {
        n < BUILD_WIDE ? rows(k_build_rows<1, false>, 1) : rows(k_build_rows<4, false>, 4);
      }
      HIPCHK(hipGetLastError());
      HIPCHK(hipStreamSynchronize(st));
      unsigned const G = nl.hstate[0], flags = nl.hstate[3];
      if (flags & OV_GHOST) {   // more ghost images than slots: grow and start again
        nl.gcap = static_cast<long>(G) + static_cast<long>(G) / 4 + 4096;
        continue;
      }
      nl.nghost = G;
      if (nl.hstate[1]) {   // a row overflowed: widen the rows and build again
        HIPCHK(hipMemcpyAsync(nl.hstate, dst, LIST_STATE * sizeof(unsigned), hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        nl.K = (static_cast<int>(nl.hstate[1]) + 15) / 16 * 16 + 16;
        continue;
      }
      bool const first = !nl.tile_seen;
      for (int l = 0; l < TILE_KINDS; ++l)
        if (all || l == level) {
          nl.tile_full[l] = nl.hstate[4 + l];
          nl.tile_used[l] = nl.hstate[8 + l];
        }
      nl.tile_seen = true;
      // A tile too full for its stage, or a first build that took the wrong form: again, with what was seen.
      if (nl.tiled && nl.tile_full[level] > TILE_MOST) continue;
      if (first && choose_tiles(nl, n, true) != level) continue;
      // The mean row, from the sample: a box is not always filled evenly.
      double const cell = nl.grid.cell[0] * nl.grid.cell[1] * nl.grid.cell[2];
      nl.mean_row = nl.hstate[12] > 0 ? 4.18879 * nl.rc * nl.rc * nl.rc / cell * nl.hstate[13] / nl.hstate[12] : mean_row(nl, n);
      // Where tiles fill the chip badly a gradient is up to 15 % faster by rows in slot order (which take a pass of
      // their own); the other passes are not (HVP at 35k to 44k atoms by tiles: 0.63 to 0.9 of the time by rows).
      // Longer rows favour the tiles (44k atoms, cut-off 6.8 A, mixed: 38.6 us by tiles at a cost of 1.6, 47 by rows).
      nl.grad_rows = nl.tiled && n < 46000 && cost > (nl.mean_row < 90.0 ? 1.3 : 1.62);
      nl.tile = tg;
      nl.tile_most = nl.tiled ? static_cast<int>(nl.tile_full[level]) : 0;
      static std::atomic<long> builds{0};
      nl.build_id = ++builds;
      nl.clear_cells = nc1;
      nl.built = true;
      return;
    }
    throw Error(FLYG_DEVICE_ERROR, "neighbour list build did not converge");
  }

  void list_update(flyg_list_s& nl, double const* d_delta, long n) {
    require(nl.built, "List::update before rebuild");
    require(n == nl.n, "Input to update has the wrong number of atoms");
    k_update<<<nblk(n, TPB), TPB, 0, nl.ctx->stream>>>(nl.pos.get(), d_delta, n, nl.rank.get(), nl.gpos.get());
    HIPCHK(hipGetLastError());
  }

  // Host-facing helpers used by the C-ABI.
  void list_positions(flyg_list_s& nl, double* d_out) {
    k_positions<<<nblk(nl.n, TPB), TPB, 0, nl.ctx->stream>>>(nl.pos.get(), nl.n, d_out);
    HIPCHK(hipGetLastError());
  }

  long list_count(flyg_list_s& nl, double rc, std::vector<int>& counts) {
    require(nl.built, "List used before rebuild");
    require(rc <= nl.rc, "r_cut is bigger than the internal r_cut");
    flyg_ctx_s& ctx = *nl.ctx;
    DBuf<int> dc;
    dc.reserve(nl.n);
    k_export<false><<<nblk(nl.n, TPB), TPB, 0, ctx.stream>>>(nl.box, rc, nl.pos.get(), nl.nbr.get(), nl.ncnt.get(), nl.K,
                                                            nl.n, nullptr, dc.get(), nullptr, nullptr, nullptr);
    counts.resize(nl.n);
    HIPCHK(hipMemcpyAsync(counts.data(), dc.get(), nl.n * sizeof(int), hipMemcpyDeviceToHost, ctx.stream));
    HIPCHK(hipStreamSynchronize(ctx.stream));
    long t = 0;
    for (int c : counts) t += c;
    return t;
  }

  void list_export(flyg_list_s& nl, double rc, int64_t* offsets, int32_t* j, int32_t* shift, double* dr) {
    std::vector<int> counts;
    long total = list_count(nl, rc, counts);
    flyg_ctx_s& ctx = *nl.ctx;
    std::vector<long long> off(nl.n + 1);
    off[0] = 0;
    for (long i = 0; i < nl.n; ++i) off[i + 1] = off[i] + counts[i];
    for (long i = 0; i <= nl.n; ++i) offsets[i] = off[i];
    DBuf<long long> doff;
    DBuf<int> dj, ds;
    DBuf<double> ddr;
    doff.reserve(nl.n + 1);
    dj.reserve(total + 1);
    ds.reserve(total + 1);
    ddr.reserve(3 * total + 3);
    HIPCHK(hipMemcpyAsync(doff.get(), off.data(), (nl.n + 1) * sizeof(long long), hipMemcpyHostToDevice, ctx.stream));
    k_export<true><<<nblk(nl.n, TPB), TPB, 0, ctx.stream>>>(nl.box, rc, nl.pos.get(), nl.nbr.get(), nl.ncnt.get(), nl.K,
                                                           nl.n, doff.get(), nullptr, dj.get(), ds.get(), ddr.get());
    HIPCHK(hipMemcpyAsync(j, dj.get(), total * sizeof(int), hipMemcpyDeviceToHost, ctx.stream));
    HIPCHK(hipMemcpyAsync(shift, ds.get(), total * sizeof(int), hipMemcpyDeviceToHost, ctx.stream));
    HIPCHK(hipMemcpyAsync(dr, ddr.get(), 3 * total * sizeof(double), hipMemcpyDeviceToHost, ctx.stream));
    HIPCHK(hipStreamSynchronize(ctx.stream));
  }

}  // namespace flyg
