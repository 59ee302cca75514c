// Device vector algebra of the plain-form minimiser, rotor and dimer: each kernel fuses the element-wise
// updates of one stage with the dot products of the next, so a chain of L-BFGS or rotor stages is one
// launch per dependent reduction.
//
// Reductions are deterministic: the grid depends on the vector length only (vec_blocks), each block
// leaves its partial sums in part[k * VMAXB + block], and whoever needs the value adds the partials in
// block order: the next kernel of the chain (every block for itself, from LDS), or the host, from a buffer
// in pinned memory that the kernel writes directly.  No block waits for another one, but in lb_newton.
//
// What bounds them: at 16k atoms (48k elements) latency, not bytes.  A launch whose last block collected
// the partials with device-scope loads in sequence took 14-16 us there, most of it that loop and its two
// device-scope fences; with the partials left to the consumer a launch takes 3 us.
#pragma once

#include "eam_host.hpp"

namespace flyg {

  constexpr int VMAXB = 240;               // most blocks of a vector kernel
  constexpr int VPART = 4 * VMAXB;         // doubles of one set of partial sums

  inline unsigned vec_blocks(long n) {     // 256 threads a block, at least 4 elements a thread
    long b = (n + 1023) / 1024;
    return static_cast<unsigned>(b < 1 ? 1 : (b > VMAXB ? VMAXB : b));
  }

  // Scalars of one device L-BFGS core.
  struct LBScalars {
    double rho[32];
    double alpha[32];
    double h0;
    unsigned stalled;   // set by a step of lb_newton that gave up, cleared by lb_first and lb_again
  };

  // The live positions of a neighbour list, moved by -u beside the kernel's own work (List::update).
  struct ListMove {
    double* pos = nullptr;    // by atom, 4 doubles each
    double* gpos = nullptr;   // by slot
    int const* rank = nullptr;
  };
  ListMove list_move(flyg_list_s& nl);

  // L-BFGS two-loop stages (lbfgs_core.cpp:29-87).  `in`: the partial sums of the stage before; `out` must
  // be another buffer.
  // First call: px = x, pg = r = g; out: r.w (w = null: r.r).
  void lb_first(flyg_ctx_s& ctx, long n, LBScalars* lb, double const* x, double const* g, double* px, double* pg, double* r,
                double const* w, double* out);
  // s = x - px, y = g - pg, px = x, pg = g; out: s.y, y.y, s.g.
  void lb_hist(flyg_ctx_s& ctx, long n, double const* x, double const* g, double* px, double* pg, double* s, double* y,
               double* out);
  // The sums of lb_hist once more, for a pair that is stored already.
  void lb_again(flyg_ctx_s& ctx, long n, LBScalars* lb, double const* s, double const* y, double const* pg, double* out);
  // alpha_j from `in` (newest: rho_j and h0 too), qout = q - alpha_j y; out: s_next.qout.
  void lb_loop1(flyg_ctx_s& ctx, long n, bool newest, int j, LBScalars* lb, double const* in, double const* q,
                double const* y, double const* s_next, double* qout, double* out);
  // The same for the oldest pair, then r = h0 (q - alpha_j y); out: y.r.
  void lb_turn(flyg_ctx_s& ctx, long n, bool newest, int j, LBScalars* lb, double const* in, double const* q,
               double const* y, double* r, double* out);
  // r += (alpha_j - rho_j in) s; out: r.w (w = null: r.r).
  void lb_loop2(flyg_ctx_s& ctx, long n, int j, LBScalars* lb, double const* in, double* r, double const* s,
                double const* w, double* out);

  // The whole two-loop in one launch, for vectors of at most NEWTON_BLOCKS blocks.  Pairs in order, oldest first (the
  // newest is written); j: their places in lb.  slots: two sets of NEWTON_SLOTS words in turn, those of `slots`
  // empty, `spare` emptied for the next call.  out: r.w (w = null: r.r).  A workgroup that polls `polls` times in vain
  // gives up: the step sets lb->stalled and *hstalled (pinned) and leaves no r and no sums.  Pair, px and pg
  // are in order all the same, so lb_again and the stage kernels can finish the step.
  constexpr int NEWTON_BLOCKS = 64;
  constexpr int NEWTON_SUMS = 2 * 32 + 3;
  constexpr int NEWTON_SLOTS = NEWTON_SUMS * NEWTON_BLOCKS;
  struct NewtonArgs {
    long n;
    int bound;
    double const* x;
    double const* g;
    double* px;
    double* pg;
    double* r;
    double const* w;
    LBScalars* lb;
    unsigned long long* slots;
    unsigned long long* spare;
    unsigned polls;
    unsigned* hstalled;
    double* out;
    double* s[32];
    double* y[32];
    int j[32];
  };
  void lb_newton(flyg_ctx_s& ctx, NewtonArgs const& a);
  void lb_empty_slots(flyg_ctx_s& ctx, unsigned long long* slots, long count);

  // Trust-region step: q *= min(1, trust / sqrt(in)), x -= q, the list follows; the sum itself goes to *hsum.  Nothing
  // happens where *stalled is set.
  void vec_step(flyg_ctx_s& ctx, long n, double trust, double const* in, double* q, double* x, ListMove lm,
                unsigned const* stalled, double* hsum);
  // out: a.b and c.d (c null: one sum); the device error flags go to *hflag (null: not copied).
  void vec_dots(flyg_ctx_s& ctx, long n, double const* a, double const* b, double const* c, double const* d, double* out,
                unsigned* hflag);
  // o = a - b; out: o.o.
  void vec_diff(flyg_ctx_s& ctx, long n, double const* a, double const* b, double* o, double* out);

  // Rotor stages (rotor.cpp:49-164).
  // delta = -dr ax, the list follows, unless *stalled is set (stalled null: always).
  void rot_offset(flyg_ctx_s& ctx, long n, double dr, double const* ax, double* delta, ListMove lm, unsigned const* stalled);
  // dg = g1 - g0; out: dg.ax.
  void rot_diff(flyg_ctx_s& ctx, long n, double const* g1, double const* g0, double const* ax, double* dg, double* out);
  // o = dg - in ax; out: the component sums of o when `sums`.
  void rot_torque(flyg_ctx_s& ctx, long n, bool sums, double const* in, double const* dg, double const* ax, double* o,
                  double* out);
  // o += mean_k (component sums `in`); out: o.o and o.w (w null: o.o alone; out null: neither).
  void vec_demean(flyg_ctx_s& ctx, long n, double mean_k, double const* in, double* o, double const* w, double* out,
                  unsigned* hflag);
  // theta -= in ax; out: theta.theta.
  void rot_orth(flyg_ctx_s& ctx, long n, double const* in, double const* ax, double* theta, double* out);
  // theta /= sqrt(in); out: dg.theta, dg.ax.
  void rot_unit(flyg_ctx_s& ctx, long n, double const* in, double* theta, double const* dg, double const* ax, double* out);
  // axp = c ax + s theta; the list moves by -dr axp - delta, delta = -dr axp.
  void rot_trial(flyg_ctx_s& ctx, long n, double c, double s, double dr, double const* ax, double const* theta, double* axp,
                 double* delta, ListMove lm);
  // out: (g1p - g0).axp.
  void rot_curv(flyg_ctx_s& ctx, long n, double const* g1p, double const* g0, double const* axp, double* out);
  // ax = c ax + s theta, g1 = w1 g1 + w2 g1p + w3 g0, dg = g1 - g0; out: dg.ax.
  void rot_accept(flyg_ctx_s& ctx, long n, double c, double s, double w1, double w2, double w3, double* ax,
                  double const* theta, double* g1, double const* g1p, double const* g0, double* dg, double* out);
  // The list moves back by delta; out: g0.ax.
  void rot_back(flyg_ctx_s& ctx, long n, double const* delta, double const* g0, double const* ax, ListMove lm, double* out);
  // eff = (g0 +) k in ax; out: the component sums of eff when `sums`, else eff.eff and eff.w (w null: none).
  void rot_eff(flyg_ctx_s& ctx, long n, bool sums, bool with_g0, double k, double const* in, double const* g0,
               double const* ax, double* eff, double const* w, double* out, unsigned* hflag);

  // Value k of a set of partial sums, added on the host (the kernel wrote them to pinned memory).
  inline double host_sum(double const* part, int k, long n) {
    double t = 0;
    for (unsigned b = 0; b < vec_blocks(n); ++b) t += part[k * VMAXB + b];
    return t;
  }

}  // namespace flyg
