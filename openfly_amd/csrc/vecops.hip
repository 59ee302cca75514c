// Vector kernels of the plain form and deterministic reductions (see vecops.hpp).
#include <cmath>

#include "vecops.hpp"

namespace flyg {

  namespace {

    constexpr int VT = 256;   // threads per block

    // Sum k of the partial sums the kernel before left, in block order, by every thread for itself.
    // `sh` holds K * VMAXB doubles; starts and ends with no barrier owed to the caller.
    template <int K>
    __device__ inline void collect(double const* __restrict__ part, double* sh, double (&tot)[K]) {
      int const nb = static_cast<int>(gridDim.x);
      for (int q = threadIdx.x; q < nb; q += VT)
#pragma unroll
        for (int k = 0; k < K; ++k) sh[k * VMAXB + q] = part[k * VMAXB + q];
      __syncthreads();
#pragma unroll
      for (int k = 0; k < K; ++k) tot[k] = 0.0;
#pragma unroll 8
      for (int b = 0; b < nb; ++b)
#pragma unroll
        for (int k = 0; k < K; ++k) tot[k] += sh[k * VMAXB + b];
    }

    // Block sums of acc[0..K) to part[k * VMAXB + block]: the wavefronts' xor trees, then the wavefronts in
    // order.
    template <int K>
    __device__ inline void leave(double const (&acc)[K], double* __restrict__ part) {
      __shared__ double sw[K][VT / 64];
      int const w = threadIdx.x >> 6;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        double const v = group_sum<64>(acc[k]);
        if ((threadIdx.x & 63) == 0) sw[k][w] = v;
      }
      __syncthreads();
      if (threadIdx.x < K) {
        double s = 0;
        for (int q = 0; q < VT / 64; ++q) s += sw[threadIdx.x][q];
        part[threadIdx.x * VMAXB + blockIdx.x] = s;
      }
    }

    // Element i of thread t of block b: i = b VT + t, then every gridDim VT further, in increasing order;
    // the loads of four elements are issued before the first of them is worked on (one after the other
    // they cost a memory round trip each).
    template <typename Load, typename Body>
    __device__ inline void vec_loop(long n, Load&& load, Body&& body) {
      long const step = static_cast<long>(gridDim.x) * VT;
      for (long i = blockIdx.x * static_cast<long>(VT) + threadIdx.x; i < n; i += 4 * step) {
        decltype(load(i)) v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (i + u * step < n) v[u] = load(i + u * step);
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (i + u * step < n) body(i + u * step, v[u]);
      }
    }

    struct V1 { double a; };
    struct V2 { double a, b; };
    struct V3 { double a, b, c; };
    struct V4 { double a, b, c, d; };
    struct V5 { double a, b, c, d, e; };

    // List::update's p -= u for one component: where it lies, and what is there.
    struct Moved {
      double p;
      long at, gat;
    };
    __device__ inline Moved to_move(ListMove const& lm, long i) {
      unsigned const a = static_cast<unsigned>(i) / 3u, c = static_cast<unsigned>(i) - 3u * a;
      Moved m;
      m.at = 4l * a + c;
      m.gat = 4l * lm.rank[a] + c;
      m.p = lm.pos[m.at];
      return m;
    }
    __device__ inline void move_one(ListMove const& lm, Moved const& m, double u) {
      double const p = m.p - u;
      lm.pos[m.at] = p;
      lm.gpos[m.gat] = p;
    }
    struct M1 { double a; Moved m; };
    struct M2 { double a, b; Moved m; };
    struct M3 { double a, b, c; Moved m; };

    // acc[i mod 3] += v without indexing registers.
    __device__ inline void add_comp(double (&acc)[3], long i, double v) {
      unsigned const c = static_cast<unsigned>(i) % 3u;
#pragma unroll
      for (unsigned k = 0; k < 3; ++k)
        if (k == c) acc[k] += v;
    }

    __global__ __launch_bounds__(VT) void k_lb_first(long n, LBScalars* __restrict__ lb, double const* __restrict__ x,
                                                     double const* __restrict__ g, double* __restrict__ px,
                                                     double* __restrict__ pg, double* __restrict__ r,
                                                     double const* __restrict__ w, double* __restrict__ out) {
      if (blockIdx.x == 0 && threadIdx.x == 0) lb->stalled = 0;
      double acc[1] = {0};
      vec_loop(
          n, [&](long i) { return V3{x[i], g[i], w ? w[i] : g[i]}; },
          [&](long i, V3 const& v) {
            px[i] = v.a;
            pg[i] = v.b;
            r[i] = v.b;
            acc[0] += v.b * v.c;
          });
      leave(acc, out);
    }

    __global__ __launch_bounds__(VT) void k_lb_hist(long n, double const* __restrict__ x, double const* __restrict__ g,
                                                    double* __restrict__ px, double* __restrict__ pg,
                                                    double* __restrict__ s, double* __restrict__ y,
                                                    double* __restrict__ out) {
      double acc[3] = {0, 0, 0};
      vec_loop(
          n, [&](long i) { return V4{x[i], g[i], px[i], pg[i]}; },
          [&](long i, V4 const& v) {
            double const si = v.a - v.c, yi = v.b - v.d;
            s[i] = si;
            y[i] = yi;
            px[i] = v.a;
            pg[i] = v.b;
            acc[0] += si * yi;
            acc[1] += yi * yi;
            acc[2] += si * v.b;
          });
      leave(acc, out);
    }

    __global__ __launch_bounds__(VT) void k_lb_again(long n, LBScalars* __restrict__ lb, double const* __restrict__ s,
                                                     double const* __restrict__ y, double const* __restrict__ pg,
                                                     double* __restrict__ out) {
      if (blockIdx.x == 0 && threadIdx.x == 0) lb->stalled = 0;
      double acc[3] = {0, 0, 0};
      vec_loop(
          n, [&](long i) { return V3{s[i], y[i], pg[i]}; },
          [&](long, V3 const& v) {
            acc[0] += v.a * v.b;
            acc[1] += v.b * v.b;
            acc[2] += v.a * v.c;
          });
      leave(acc, out);
    }

    // alpha_j of loop 1 from the stage before; the newest pair's rho and h0 come from lb_hist's sums.
    template <bool NEWEST>
    __device__ inline double alpha_of(double const* __restrict__ in, double* sh, LBScalars* __restrict__ lb, int j,
                                      double& h0) {
      double alpha;
      if constexpr (NEWEST) {
        double t[3];
        collect(in, sh, t);
        double const rho = 1.0 / fabs(t[0]);
        h0 = (1.0 / rho) / t[1];
        alpha = rho * t[2];
        if (blockIdx.x == 0 && threadIdx.x == 0) {
          lb->rho[j] = rho;
          lb->h0 = h0;
        }
      } else {
        double t[1];
        collect(in, sh, t);
        alpha = lb->rho[j] * t[0];
        h0 = lb->h0;
      }
      if (blockIdx.x == 0 && threadIdx.x == 0) lb->alpha[j] = alpha;
      return alpha;
    }

    template <bool NEWEST>
    __global__ __launch_bounds__(VT) void k_lb_loop1(long n, int j, LBScalars* __restrict__ lb, double const* __restrict__ in,
                                                     double const* q, double const* __restrict__ y,
                                                     double const* __restrict__ s_next, double* qout,
                                                     double* __restrict__ out) {
      __shared__ double sh[3 * VMAXB];
      double h0;
      double const c = -1.0 * alpha_of<NEWEST>(in, sh, lb, j, h0);
      double acc[1] = {0};
      vec_loop(
          n, [&](long i) { return V3{q[i], y[i], s_next[i]}; },
          [&](long i, V3 const& v) {
            double o = v.a;
            o += c * v.b;
            qout[i] = o;
            acc[0] += v.c * o;
          });
      leave(acc, out);
    }

    template <bool NEWEST>
    __global__ __launch_bounds__(VT) void k_lb_turn(long n, int j, LBScalars* __restrict__ lb, double const* __restrict__ in,
                                                    double const* __restrict__ q, double const* __restrict__ y,
                                                    double* __restrict__ r, double* __restrict__ out) {
      __shared__ double sh[3 * VMAXB];
      double h0;
      double const c = -1.0 * alpha_of<NEWEST>(in, sh, lb, j, h0);
      double acc[1] = {0};
      vec_loop(
          n, [&](long i) { return V2{q[i], y[i]}; },
          [&](long i, V2 const& v) {
            double o = v.a;
            o += c * v.b;
            double const ri = h0 * o;
            r[i] = ri;
            acc[0] += v.b * ri;
          });
      leave(acc, out);
    }

    __global__ __launch_bounds__(VT) void k_lb_loop2(long n, int j, LBScalars const* __restrict__ lb,
                                                     double const* __restrict__ in, double* __restrict__ r,
                                                     double const* __restrict__ s, double const* __restrict__ w,
                                                     double* __restrict__ out) {
      __shared__ double sh[VMAXB];
      double t[1];
      collect(in, sh, t);
      double const c = lb->alpha[j] - lb->rho[j] * t[0];
      double acc[1] = {0};
      vec_loop(
          n, [&](long i) { return V3{r[i], s[i], w ? w[i] : 0.0}; },
          [&](long i, V3 const& v) {
            double o = v.a;
            o += c * v.b;
            r[i] = o;
            acc[0] += o * (w ? v.c : o);
          });
      leave(acc, out);
    }

    // ---- The two-loop in one launch ------------------------------------------------------------------
    // Its 2 m sums are a chain, each needed by every element before the next.  As launches a link costs 3.6 us at
    // 65k elements (an empty launch 2.35); here it is a store and a poll through the device's memory, 1.1 us at 3k
    // elements, 2.8 at 30k and 3.5 at 65k, where the two meet (NEWTON_BLOCKS).  A
    // thread keeps its (at most four) elements of q and r in registers from the first stage to the last, so no
    // vector data crosses workgroups, only partial sums do: a workgroup writes its sum to a slot of its own, and one
    // wavefront of every workgroup reads all of them until none is empty.  An empty slot holds a
    // signalling NaN, which no sum can be.  Sums and expressions are those of the stage kernels: the same bits.
    // Every workgroup must be resident at once.  At most NEWTON_BLOCKS = 64 of 256 threads are launched, on a chip that
    // holds 2048; but long kernels of other streams (the search server's) can leave no room for some of them until
    // they end.  So the wait is bounded, by polls and not by the clock, which runs on while a queue is switched
    // out: a workgroup that polls in vain stops waiting, the step is marked as given up, and every workgroup
    // runs to its end, publishing its sums on the way so that nobody waits for it.  What the step writes besides r
    // and the sums (px, pg, the newest pair) does not depend on them, so the caller finishes it by stage kernels.
    constexpr unsigned long long EMPTY_SLOT = 0x7ff4deadbeef0badull;

    __global__ void k_empty_slots(unsigned long long* slots, long count) {
      long const i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
      if (i < count) slots[i] = EMPTY_SLOT;
    }

    struct NewtonLds {
      double sw[3][VT / 64];
      double sh[3][NEWTON_BLOCKS];
      double alpha[32], rho[32];
      int dead;
    };

    // Totals over the grid of acc[0..K), by sum numbers id .. id + K - 1.
    template <int K>
    __device__ inline void grid_sum(NewtonArgs const& A, NewtonLds& L, int id, double const (&acc)[K], double (&tot)[K]) {
      int const nb = static_cast<int>(gridDim.x), w = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        double const v = group_sum<64>(acc[k]);
        if (lane == 0) L.sw[k][w] = v;
      }
      __syncthreads();
      if (threadIdx.x < K) {
        double s = 0;
        for (int q = 0; q < VT / 64; ++q) s += L.sw[threadIdx.x][q];
        __hip_atomic_store(&A.slots[(id + threadIdx.x) * NEWTON_BLOCKS + blockIdx.x],
                           static_cast<unsigned long long>(__double_as_longlong(s)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      if (w == 0) {
        unsigned polls = 0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
          unsigned long long const* slot = &A.slots[(id + k) * NEWTON_BLOCKS + (lane < nb ? lane : 0)];
          unsigned long long v;
          while (true) {   // ends when every slot is filled or after `polls` rounds
            v = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (__all(v != EMPTY_SLOT) || L.dead) break;
            if (++polls > A.polls) {
              L.dead = 1;
              break;
            }
            __builtin_amdgcn_s_sleep(1);   // 64 clocks, as the clock that was read here before took
          }
          L.sh[k][lane] = __longlong_as_double(static_cast<long long>(v));
        }
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < K; ++k) tot[k] = 0.0;
#pragma unroll 8
      for (int b = 0; b < nb; ++b)
#pragma unroll
        for (int k = 0; k < K; ++k) tot[k] += L.sh[k][b];
    }

    __global__ __launch_bounds__(VT) void k_lb_newton(NewtonArgs A) {
      __shared__ NewtonLds L;
      long const step = static_cast<long>(gridDim.x) * VT;
      long const i0 = blockIdx.x * static_cast<long>(VT) + threadIdx.x;
      int const bound = A.bound;
      for (int q = threadIdx.x; q < NEWTON_SUMS; q += VT) A.spare[q * NEWTON_BLOCKS + blockIdx.x] = EMPTY_SLOT;
      if (threadIdx.x == 0) L.dead = A.polls == 0;   // told not to wait
      if (threadIdx.x < bound - 1) L.rho[threadIdx.x] = A.lb->rho[A.j[threadIdx.x]];
      auto load = [&](double const* p, double (&v)[4]) {
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = i0 + u * step < A.n ? p[i0 + u * step] : 0.0;
      };
      double q[4], y[4], s[4], yn[4];   // q, later r; the pair's y; s and y of the stage to come
      double acc[1], tot[1];
      double h0;
      {
        double x[4], px[4], pg[4], acc3[3] = {0, 0, 0}, t[3];
        load(A.x, x);
        load(A.g, q);
        load(A.px, px);
        load(A.pg, pg);
        if (bound > 1) {
          load(A.s[bound - 2], s);
          load(A.y[bound - 2], yn);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          long const i = i0 + u * step;
          if (i < A.n) {
            double const si = x[u] - px[u], yi = q[u] - pg[u];
            A.s[bound - 1][i] = si;
            A.y[bound - 1][i] = yi;
            A.px[i] = x[u];
            A.pg[i] = q[u];
            acc3[0] += si * yi;
            acc3[1] += yi * yi;
            acc3[2] += si * q[u];
            y[u] = yi;
          }
        }
        grid_sum<3>(A, L, 0, acc3, t);
        double const rho = 1.0 / fabs(t[0]);
        h0 = (1.0 / rho) / t[1];
        tot[0] = rho * t[2];   // alpha of the newest pair
        if (threadIdx.x == 0) {
          L.rho[bound - 1] = rho;
          if (blockIdx.x == 0) {
            A.lb->rho[A.j[bound - 1]] = rho;
            A.lb->h0 = h0;
          }
        }
      }
      int id = 3;
      double alpha = tot[0];
      for (int i = bound - 1; i > 0; --i) {   // loop 1, newest to oldest; s, yn: pair i - 1
        if (threadIdx.x == 0) L.alpha[i] = alpha;
        double const c = -1.0 * alpha;
        acc[0] = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (i0 + u * step < A.n) {
            double o = q[u];
            o += c * y[u];
            q[u] = o;
            acc[0] += s[u] * o;
          }
#pragma unroll
        for (int u = 0; u < 4; ++u) y[u] = yn[u];
        if (i > 1) {
          load(A.s[i - 2], s);
          load(A.y[i - 2], yn);
        }
        grid_sum<1>(A, L, id++, acc, tot);
        alpha = L.rho[i - 1] * tot[0];
      }
      if (threadIdx.x == 0) L.alpha[0] = alpha;
      {
        double const c = -1.0 * alpha;
        acc[0] = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (i0 + u * step < A.n) {
            double o = q[u];
            o += c * y[u];
            double const ri = h0 * o;
            q[u] = ri;
            acc[0] += y[u] * ri;
          }
      }
      for (int i = 0; i < bound; ++i) {   // loop 2, oldest to newest
        load(A.s[i], s);
        bool const last = i + 1 == bound;
        if (!last) {
          load(A.y[i + 1], yn);
        } else if (A.w) {
          load(A.w, yn);
        }
        grid_sum<1>(A, L, id++, acc, tot);
        double const al = L.alpha[i], rho = L.rho[i];
        double const c = al - rho * tot[0];
        acc[0] = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (i0 + u * step < A.n) {
            double o = q[u];
            o += c * s[u];
            q[u] = o;
            acc[0] += o * (last && !A.w ? o : yn[u]);
          }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (i0 + u * step < A.n) A.r[i0 + u * step] = q[u];
      leave(acc, A.out);
      if (threadIdx.x == 0 && L.dead) {
        __hip_atomic_store(&A.lb->stalled, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(A.hstalled, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }

    __global__ __launch_bounds__(VT) void k_step(long n, double trust, double const* __restrict__ in, double* __restrict__ q,
                                                 double* __restrict__ x, ListMove lm, unsigned const* __restrict__ stalled,
                                                 double* __restrict__ hsum) {
      __shared__ double sh[VMAXB];
      double t[1];
      unsigned const off = *stalled;   // its load is under way with the sums'
      collect(in, sh, t);
      if (off) return;
      if (blockIdx.x == 0 && threadIdx.x == 0) *hsum = t[0];
      double const c = fmin(1.0, trust / sqrt(t[0]));
      vec_loop(
          n, [&](long i) { return M2{q[i], x[i], to_move(lm, i)}; },
          [&](long i, M2 const& v) {
            double const o = c * v.a;
            q[i] = o;
            x[i] = v.b - o;
            move_one(lm, v.m, o);
          });
    }

    __global__ __launch_bounds__(VT) void k_dots(long n, double const* __restrict__ a, double const* __restrict__ b,
                                                 double const* __restrict__ c, double const* __restrict__ d,
                                                 double* __restrict__ out, unsigned const* __restrict__ flags,
                                                 unsigned* __restrict__ hflag) {
      double acc[2] = {0, 0};
      vec_loop(
          n, [&](long i) { return V4{a[i], b[i], c ? c[i] : 0.0, c ? d[i] : 0.0}; },
          [&](long, V4 const& v) {
            acc[0] += v.a * v.b;
            acc[1] += v.c * v.d;
          });
      leave(acc, out);
      if (hflag && blockIdx.x == 0 && threadIdx.x == 0) *hflag = *flags;
    }

    __global__ __launch_bounds__(VT) void k_diff(long n, double const* __restrict__ a, double const* __restrict__ b,
                                                 double* __restrict__ o, double* __restrict__ out) {
      double acc[1] = {0};
      vec_loop(
          n, [&](long i) { return V2{a[i], b[i]}; },
          [&](long i, V2 const& w) {
            double const v = w.a - w.b;
            o[i] = v;
            acc[0] += v * v;
          });
      leave(acc, out);
    }

    __global__ __launch_bounds__(VT) void k_rot_offset(long n, double dr, double const* __restrict__ ax,
                                                       double* __restrict__ delta, ListMove lm,
                                                       unsigned const* __restrict__ stalled) {
      bool const move = !stalled || !*stalled;
      vec_loop(
          n, [&](long i) { return M1{ax[i], to_move(lm, i)}; },
          [&](long i, M1 const& v) {
            double const o = -dr * v.a;
            delta[i] = o;
            if (move) move_one(lm, v.m, o);
          });
    }

    __global__ __launch_bounds__(VT) void k_rot_diff(long n, double const* __restrict__ g1, double const* __restrict__ g0,
                                                     double const* __restrict__ ax, double* __restrict__ dg,
                                                     double* __restrict__ out) {
      double acc[1] = {0};
      vec_loop(
          n, [&](long i) { return V3{g1[i], g0[i], ax[i]}; },
          [&](long i, V3 const& v) {
            double const o = v.a - v.b;
            dg[i] = o;
            acc[0] += o * v.c;
          });
      leave(acc, out);
    }

    template <bool SUMS>
    __global__ __launch_bounds__(VT) void k_rot_torque(long n, double const* __restrict__ in, double const* __restrict__ dg,
                                                       double const* __restrict__ ax, double* __restrict__ o,
                                                       double* __restrict__ out) {
      __shared__ double sh[VMAXB];
      double t[1];
      collect(in, sh, t);
      double const c = -1.0 * t[0];
      double acc[3] = {0, 0, 0};
      vec_loop(
          n, [&](long i) { return V2{dg[i], ax[i]}; },
          [&](long i, V2 const& w) {
            double v = w.a;
            v += c * w.b;
            o[i] = v;
            if (SUMS) add_comp(acc, i, v);
          });
      if (SUMS) leave(acc, out);
    }

    __global__ __launch_bounds__(VT) void k_demean(long n, double mean_k, double const* __restrict__ in,
                                                   double* __restrict__ o, double const* __restrict__ w,
                                                   double* __restrict__ out, unsigned const* __restrict__ flags,
                                                   unsigned* __restrict__ hflag) {
      __shared__ double sh[3 * VMAXB];
      double t[3];
      collect(in, sh, t);
      double const m0 = mean_k * t[0], m1 = mean_k * t[1], m2 = mean_k * t[2];
      double acc[2] = {0, 0};
      vec_loop(
          n, [&](long i) { return V2{o[i], w ? w[i] : 0.0}; },
          [&](long i, V2 const& e) {
            unsigned const c = static_cast<unsigned>(i) % 3u;
            double const v = e.a + (c == 0 ? m0 : (c == 1 ? m1 : m2));
            o[i] = v;
            acc[0] += v * v;
            acc[1] += v * e.b;
          });
      if (out) leave(acc, out);
      if (hflag && blockIdx.x == 0 && threadIdx.x == 0) *hflag = *flags;
    }

    __global__ __launch_bounds__(VT) void k_rot_orth(long n, double const* __restrict__ in, double const* __restrict__ ax,
                                                     double* __restrict__ theta, double* __restrict__ out) {
      __shared__ double sh[VMAXB];
      double t[1];
      collect(in, sh, t);
      double const c = -1.0 * t[0];
      double acc[1] = {0};
      vec_loop(
          n, [&](long i) { return V2{theta[i], ax[i]}; },
          [&](long i, V2 const& v) {
            double o = v.a;
            o += c * v.b;
            theta[i] = o;
            acc[0] += o * o;
          });
      leave(acc, out);
    }

    __global__ __launch_bounds__(VT) void k_rot_unit(long n, double const* __restrict__ in, double* __restrict__ theta,
                                                     double const* __restrict__ dg, double const* __restrict__ ax,
                                                     double* __restrict__ out) {
      __shared__ double sh[VMAXB];
      double t[1];
      collect(in, sh, t);
      double const c = 1.0 / sqrt(t[0]);
      double acc[2] = {0, 0};
      vec_loop(
          n, [&](long i) { return V3{theta[i], dg[i], ax[i]}; },
          [&](long i, V3 const& v) {
            double const o = c * v.a;
            theta[i] = o;
            acc[0] += v.b * o;
            acc[1] += v.b * v.c;
          });
      leave(acc, out);
    }

    __global__ __launch_bounds__(VT) void k_rot_trial(long n, double c, double s, double dr, double const* __restrict__ ax,
                                                      double const* __restrict__ theta, double* __restrict__ axp,
                                                      double* __restrict__ delta, ListMove lm) {
      vec_loop(
          n, [&](long i) { return M3{ax[i], theta[i], delta[i], to_move(lm, i)}; },
          [&](long i, M3 const& v) {
            double o = c * v.a;
            o += s * v.b;
            axp[i] = o;
            double const e = -dr * o;
            delta[i] = e;
            move_one(lm, v.m, e - v.c);
          });
    }

    __global__ __launch_bounds__(VT) void k_rot_curv(long n, double const* __restrict__ g1p, double const* __restrict__ g0,
                                                     double const* __restrict__ axp, double* __restrict__ out) {
      double acc[1] = {0};
      vec_loop(
          n, [&](long i) { return V3{g1p[i], g0[i], axp[i]}; },
          [&](long, V3 const& v) {
            double const o = v.a - v.b;
            acc[0] += o * v.c;
          });
      leave(acc, out);
    }

    __global__ __launch_bounds__(VT) void k_rot_accept(long n, double c, double s, double w1, double w2, double w3,
                                                       double* __restrict__ ax, double const* __restrict__ theta,
                                                       double* __restrict__ g1, double const* __restrict__ g1p,
                                                       double const* __restrict__ g0, double* __restrict__ dg,
                                                       double* __restrict__ out) {
      double acc[1] = {0};
      vec_loop(
          n, [&](long i) { return V5{ax[i], theta[i], g1[i], g1p[i], g0[i]}; },
          [&](long i, V5 const& v) {
            double a = c * v.a;
            a += s * v.b;
            ax[i] = a;
            double o = w1 * v.c;
            o += w2 * v.d;
            o += w3 * v.e;
            g1[i] = o;
            double const d = o - v.e;
            dg[i] = d;
            acc[0] += d * a;
          });
      leave(acc, out);
    }

    __global__ __launch_bounds__(VT) void k_rot_back(long n, double const* __restrict__ delta, double const* __restrict__ g0,
                                                     double const* __restrict__ ax, ListMove lm, double* __restrict__ out) {
      double acc[1] = {0};
      vec_loop(
          n, [&](long i) { return M3{delta[i], g0[i], ax[i], to_move(lm, i)}; },
          [&](long, M3 const& v) {
            move_one(lm, v.m, -v.a);
            acc[0] += v.b * v.c;
          });
      leave(acc, out);
    }

    template <bool SUMS, bool G0>
    __global__ __launch_bounds__(VT) void k_rot_eff(long n, double k, double const* __restrict__ in,
                                                    double const* __restrict__ g0, double const* __restrict__ ax,
                                                    double* __restrict__ eff, double const* __restrict__ w,
                                                    double* __restrict__ out, unsigned const* __restrict__ flags,
                                                    unsigned* __restrict__ hflag) {
      __shared__ double sh[VMAXB];
      double t[1];
      collect(in, sh, t);
      double const c = k * t[0];
      double acc[3] = {0, 0, 0};
      vec_loop(
          n, [&](long i) { return V3{G0 ? g0[i] : 0.0, ax[i], w ? w[i] : 0.0}; },
          [&](long i, V3 const& v) {
            double o;
            if (G0) {
              o = v.a;
              o += c * v.b;
            } else {
              o = c * v.b;
            }
            eff[i] = o;
            if (SUMS) {
              add_comp(acc, i, o);
            } else {
              acc[0] += o * o;
              acc[1] += o * v.c;
            }
          });
      leave(acc, out);
      if (hflag && blockIdx.x == 0 && threadIdx.x == 0) *hflag = *flags;
    }

    __global__ __launch_bounds__(VT) void k_sum(double const* __restrict__ x, long n, double* __restrict__ out,
                                                unsigned const* __restrict__ flags, unsigned* __restrict__ hflag) {
      double acc[1] = {0};
      vec_loop(
          n, [&](long i) { return V1{x[i]}; }, [&](long, V1 const& v) { acc[0] += v.a; });
      leave(acc, out);
      if (hflag && blockIdx.x == 0 && threadIdx.x == 0) *hflag = *flags;
    }

  }  // namespace

#define FLYG_VEC_LAUNCH(kernel, ...) \
  kernel<<<vec_blocks(n), VT, 0, ctx.stream>>>(n, __VA_ARGS__); \
  HIPCHK(hipGetLastError())

  ListMove list_move(flyg_list_s& nl) {
    return ListMove{reinterpret_cast<double*>(nl.pos.get()), reinterpret_cast<double*>(nl.gpos.get()), nl.rank.get()};
  }

  void lb_first(flyg_ctx_s& ctx, long n, LBScalars* lb, double const* x, double const* g, double* px, double* pg, double* r,
                double const* w, double* out) {
    FLYG_VEC_LAUNCH(k_lb_first, lb, x, g, px, pg, r, w, out);
  }
  void lb_again(flyg_ctx_s& ctx, long n, LBScalars* lb, double const* s, double const* y, double const* pg, double* out) {
    FLYG_VEC_LAUNCH(k_lb_again, lb, s, y, pg, out);
  }
  void lb_hist(flyg_ctx_s& ctx, long n, double const* x, double const* g, double* px, double* pg, double* s, double* y,
               double* out) {
    FLYG_VEC_LAUNCH(k_lb_hist, x, g, px, pg, s, y, out);
  }
  void lb_loop1(flyg_ctx_s& ctx, long n, bool newest, int j, LBScalars* lb, double const* in, double const* q,
                double const* y, double const* s_next, double* qout, double* out) {
    if (newest) {
      FLYG_VEC_LAUNCH(k_lb_loop1<true>, j, lb, in, q, y, s_next, qout, out);
    } else {
      FLYG_VEC_LAUNCH(k_lb_loop1<false>, j, lb, in, q, y, s_next, qout, out);
    }
  }
  void lb_turn(flyg_ctx_s& ctx, long n, bool newest, int j, LBScalars* lb, double const* in, double const* q,
               double const* y, double* r, double* out) {
    if (newest) {
      FLYG_VEC_LAUNCH(k_lb_turn<true>, j, lb, in, q, y, r, out);
    } else {
      FLYG_VEC_LAUNCH(k_lb_turn<false>, j, lb, in, q, y, r, out);
    }
  }
  void lb_loop2(flyg_ctx_s& ctx, long n, int j, LBScalars* lb, double const* in, double* r, double const* s,
                double const* w, double* out) {
    FLYG_VEC_LAUNCH(k_lb_loop2, j, lb, in, r, s, w, out);
  }
  void lb_newton(flyg_ctx_s& ctx, NewtonArgs const& a) {
    k_lb_newton<<<vec_blocks(a.n), VT, 0, ctx.stream>>>(a);
    HIPCHK(hipGetLastError());
  }
  void lb_empty_slots(flyg_ctx_s& ctx, unsigned long long* slots, long count) {
    k_empty_slots<<<static_cast<unsigned>((count + VT - 1) / VT), VT, 0, ctx.stream>>>(slots, count);
    HIPCHK(hipGetLastError());
  }
  void vec_step(flyg_ctx_s& ctx, long n, double trust, double const* in, double* q, double* x, ListMove lm,
                unsigned const* stalled, double* hsum) {
    FLYG_VEC_LAUNCH(k_step, trust, in, q, x, lm, stalled, hsum);
  }
  void vec_dots(flyg_ctx_s& ctx, long n, double const* a, double const* b, double const* c, double const* d, double* out,
                unsigned* hflag) {
    FLYG_VEC_LAUNCH(k_dots, a, b, c, d, out, ctx.dflags.get(), hflag);
  }
  void vec_diff(flyg_ctx_s& ctx, long n, double const* a, double const* b, double* o, double* out) {
    FLYG_VEC_LAUNCH(k_diff, a, b, o, out);
  }
  void rot_offset(flyg_ctx_s& ctx, long n, double dr, double const* ax, double* delta, ListMove lm, unsigned const* stalled) {
    FLYG_VEC_LAUNCH(k_rot_offset, dr, ax, delta, lm, stalled);
  }
  void rot_diff(flyg_ctx_s& ctx, long n, double const* g1, double const* g0, double const* ax, double* dg, double* out) {
    FLYG_VEC_LAUNCH(k_rot_diff, g1, g0, ax, dg, out);
  }
  void rot_torque(flyg_ctx_s& ctx, long n, bool sums, double const* in, double const* dg, double const* ax, double* o,
                  double* out) {
    if (sums) {
      FLYG_VEC_LAUNCH(k_rot_torque<true>, in, dg, ax, o, out);
    } else {
      FLYG_VEC_LAUNCH(k_rot_torque<false>, in, dg, ax, o, out);
    }
  }
  void vec_demean(flyg_ctx_s& ctx, long n, double mean_k, double const* in, double* o, double const* w, double* out,
                  unsigned* hflag) {
    FLYG_VEC_LAUNCH(k_demean, mean_k, in, o, w, out, ctx.dflags.get(), hflag);
  }
  void rot_orth(flyg_ctx_s& ctx, long n, double const* in, double const* ax, double* theta, double* out) {
    FLYG_VEC_LAUNCH(k_rot_orth, in, ax, theta, out);
  }
  void rot_unit(flyg_ctx_s& ctx, long n, double const* in, double* theta, double const* dg, double const* ax, double* out) {
    FLYG_VEC_LAUNCH(k_rot_unit, in, theta, dg, ax, out);
  }
  void rot_trial(flyg_ctx_s& ctx, long n, double c, double s, double dr, double const* ax, double const* theta, double* axp,
                 double* delta, ListMove lm) {
    FLYG_VEC_LAUNCH(k_rot_trial, c, s, dr, ax, theta, axp, delta, lm);
  }
  void rot_curv(flyg_ctx_s& ctx, long n, double const* g1p, double const* g0, double const* axp, double* out) {
    FLYG_VEC_LAUNCH(k_rot_curv, g1p, g0, axp, out);
  }
  void rot_accept(flyg_ctx_s& ctx, long n, double c, double s, double w1, double w2, double w3, double* ax,
                  double const* theta, double* g1, double const* g1p, double const* g0, double* dg, double* out) {
    FLYG_VEC_LAUNCH(k_rot_accept, c, s, w1, w2, w3, ax, theta, g1, g1p, g0, dg, out);
  }
  void rot_back(flyg_ctx_s& ctx, long n, double const* delta, double const* g0, double const* ax, ListMove lm, double* out) {
    FLYG_VEC_LAUNCH(k_rot_back, delta, g0, ax, lm, out);
  }
  void rot_eff(flyg_ctx_s& ctx, long n, bool sums, bool with_g0, double k, double const* in, double const* g0,
               double const* ax, double* eff, double const* w, double* out, unsigned* hflag) {
    unsigned const* fl = ctx.dflags.get();
    if (sums && with_g0) {
      FLYG_VEC_LAUNCH((k_rot_eff<true, true>), k, in, g0, ax, eff, w, out, fl, hflag);
    } else if (sums) {
      FLYG_VEC_LAUNCH((k_rot_eff<true, false>), k, in, g0, ax, eff, w, out, fl, hflag);
    } else if (with_g0) {
      FLYG_VEC_LAUNCH((k_rot_eff<false, true>), k, in, g0, ax, eff, w, out, fl, hflag);
    } else {
      FLYG_VEC_LAUNCH((k_rot_eff<false, false>), k, in, g0, ax, eff, w, out, fl, hflag);
    }
  }

  void dev_sum(flyg_ctx_s& ctx, double const* x, long n, double* part, unsigned* hflag) {
    k_sum<<<vec_blocks(n), VT, 0, ctx.stream>>>(x, n, part, ctx.dflags.get(), hflag);
    HIPCHK(hipGetLastError());
  }

}  // namespace flyg
