// Plain-form StepLBFGS, LBFGS::minimise, Rotor::eff_gradient and Dimer::find_sp (FP64).
//
// Control flow restates lbfgs_core.cpp:29-87, lbfgs.cpp:29-115, rotor.cpp:33-164 and dimer.cpp:28-171;
// scalars that steer the host-side control flow (norms, curvatures, projections) are read back once
// per decision, everything else stays on the device.
#include <cmath>
#include <utility>

#include "plain.hpp"

namespace flyg {

  namespace {
    void copy(flyg_ctx_s& ctx, double* dst, double const* src, long n) {
      HIPCHK(hipMemcpyAsync(dst, src, n * sizeof(double), hipMemcpyDeviceToDevice, ctx.stream));
    }

    // Options::fout of the reference (lbfgs.cpp:75-77, dimer.cpp:88-90): the positions at the start of
    // iteration `it`, copied to the host, go to the caller's observer.
    void observe(flyg_ctx_s& ctx, flyg_step_observer fn, void* user, int it, double const* d_x, long n,
                 std::vector<double>& host) {
      if (!fn) return;
      host.resize(static_cast<std::size_t>(3 * n));
      HIPCHK(hipMemcpyAsync(host.data(), d_x, 3 * n * sizeof(double), hipMemcpyDeviceToHost, ctx.stream));
      HIPCHK(hipStreamSynchronize(ctx.stream));
      if (int const rc = fn(user, it, host.data(), n)) {
        throw Error(FLYG_STOPPED, "the step observer stopped the run at iteration " + std::to_string(it) +
                                      " (returned " + std::to_string(rc) + ")");
      }
    }
  }  // namespace

  // ================================================================================================
  // DevLBFGS (two-loop recursion, Nocedal & Wright Alg. 7.4; rho = 1/|s.y|; H0 = (1/rho)/(y.y) from the
  // newest pair; the first call returns g).
  // ================================================================================================

  DevLBFGS::DevLBFGS(flyg_ctx_s* ctx, int m, bool rotor)
      : m_ctx(ctx), m_hstalled(ctx->hflags + (rotor ? 4 : 3)), m_m(m), m_s(static_cast<std::size_t>(m)), m_y(static_cast<std::size_t>(m)) {
    require(m > 0 && m <= 32, "L-BFGS history length must be in [1, 32]");
    m_sc.reserve(1);
    m_part.reserve(2 * VPART);
  }

  double* DevLBFGS::newton_step(double const* x, double const* g, long N, double const* w, double const** sums,
                                bool may_wait) {
    flyg_ctx_s& ctx = *m_ctx;
    if (m_k > 0) require(N == m_N, "Call to newton_step() with a different number of atoms than the history");
    if (N != m_N) {
      for (auto& v : m_s) v.p(N);
      for (auto& v : m_y) v.p(N);
      m_px.p(N);
      m_pg.p(N);
      m_q.p(N);
      m_r.p(N);
      m_N = N;
    }
    LBScalars* lb = m_sc.get();
    double* out = m_part.get() + VPART;
    double* r = m_r.get();
    if (m_k == 0) {
      lb_first(ctx, N, lb, x, g, m_px.get(), m_pg.get(), r, w, out);
      ++m_k;
      if (sums) *sums = out;
      return r;
    }
    int const bound = m_k <= m_m ? m_k : m_m;
    // One launch, for longer vectors a launch a stage.
    if (may_wait && vec_blocks(N) <= NEWTON_BLOCKS && m_rest == 0) {
      if (m_slots_n != N) {
        m_slots.reserve(2 * NEWTON_SLOTS);
        lb_empty_slots(ctx, m_slots.get(), 2 * NEWTON_SLOTS);
      }
      m_slots_n = -1;   // until the launch has succeeded
      NewtonArgs a{};
      a.n = N;
      a.bound = bound;
      a.x = x;
      a.g = g;
      a.px = m_px.get();
      a.pg = m_pg.get();
      a.r = r;
      a.w = w;
      a.lb = lb;
      a.slots = m_slots.get() + m_slots_used * NEWTON_SLOTS;
      m_slots_used = 1 - m_slots_used;
      a.spare = m_slots.get() + m_slots_used * NEWTON_SLOTS;
      a.polls = ctx.step_polls;
      a.hstalled = m_hstalled;
      a.out = out;
      for (int i = 0; i < bound; ++i) {
        a.j[i] = pair(m_k, i);
        a.s[i] = m_s[a.j[i]].get();
        a.y[i] = m_y[a.j[i]].get();
      }
      *m_hstalled = 0;
      lb_newton(ctx, a);
      m_slots_n = N;
      ++m_k;
      if (sums) *sums = out;
      return r;
    }
    if (m_rest > 0) --m_rest;
    int const newest = pair(m_k, bound - 1);
    lb_hist(ctx, N, x, g, m_px.get(), m_pg.get(), m_s[newest].get(), m_y[newest].get(), out);
    ++m_k;
    return stages(m_k - 1, w, sums);
  }

  // The step of call k + 1 from the sums that lb_hist left, a launch a stage.
  double* DevLBFGS::stages(int k, double const* w, double const** sums) {
    flyg_ctx_s& ctx = *m_ctx;
    long const N = m_N;
    LBScalars* lb = m_sc.get();
    double* out = m_part.get();         // partial sums of this stage
    double* in = out + VPART;           // ... and of the one before
    double* q = m_q.get();
    double* r = m_r.get();
    int const bound = k <= m_m ? k : m_m;
    int const newest = pair(k, bound - 1);
    double const* from = m_pg.get();    // q before loop 1: the gradient lb_hist kept
    for (int i = bound - 1; i > 0; --i) {
      int const j = pair(k, i);
      lb_loop1(ctx, N, j == newest, j, lb, in, from, m_y[j].get(), m_s[pair(k, i - 1)].get(), q, out);
      std::swap(in, out);
      from = q;
    }
    int const oldest = pair(k, 0);
    lb_turn(ctx, N, bound == 1, oldest, lb, in, from, m_y[oldest].get(), r, out);
    std::swap(in, out);
    for (int i = 0; i < bound; ++i) {
      int const j = pair(k, i);
      lb_loop2(ctx, N, j, lb, in, r, m_s[j].get(), i + 1 < bound ? m_y[pair(k, i + 1)].get() : w, out);
      std::swap(in, out);
    }
    if (sums) *sums = in;
    return r;
  }

  bool DevLBFGS::stalled() {
    bool const s = *m_hstalled != 0;
    *m_hstalled = 0;
    return s;
  }

  double* DevLBFGS::again(double const* w, double const** sums) {
    int const k = m_k - 1, newest = pair(k, (k <= m_m ? k : m_m) - 1);
    m_rest = m_ctx->step_polls / 64;   // the chip is busy: a wait in vain is spread over so many steps
    lb_again(*m_ctx, m_N, m_sc.get(), m_s[newest].get(), m_y[newest].get(), m_pg.get(), m_part.get() + VPART);
    return stages(k, w, sums);
  }

  std::unique_ptr<flyg_list_s> make_list(flyg_ctx_s* ctx, double const* basis, int const* periodic, double rc) {
    auto nl = std::make_unique<flyg_list_s>();
    nl->ctx = ctx;
    nl->box = make_box(basis, periodic);
    nl->grid = make_grid(nl->box, rc);
    nl->rc = rc;
    return nl;
  }

  namespace {
    void check_flags(flyg_ctx_s& ctx) { throw_flags(ctx.take_flags()); }

    void sync(flyg_ctx_s& ctx) { HIPCHK(hipStreamSynchronize(ctx.stream)); }

    // After a kernel that wrote its sums and the error flags to pinned memory.
    void sync_checked(flyg_ctx_s& ctx) {
      sync(ctx);
      if (ctx.hflags[1]) check_flags(ctx);
    }
  }  // namespace

  // ================================================================================================
  // LBFGS::minimise (lbfgs.cpp:29-115)
  // ================================================================================================

  bool lbfgs_minimise(flyg_lbfgs_s& m, flyg_eam_s& e, double* d_pos, double* d_grad, uint32_t const* d_types,
                      uint8_t const* d_frozen, long n, int* iterations) {
    flyg_ctx_s& ctx = *m.ctx;
    flyg_lbfgs_options const& o = m.opt;
    long N = 3 * n;
    double skin = std::fmax(std::pow(o.skin_frac, 1. / 3.) - 1, 0.0) * e.tab.rc;
    double rc = e.tab.rc + skin;
    if (!m.nl || m.nl->rc != rc) m.nl = make_list(&ctx, m.basis, m.periodic, rc);
    if (!m.core) m.core = std::make_unique<DevLBFGS>(&ctx, o.n);
    m.core->clear();
    double* x = d_pos;
    double* g = d_grad;
    double* hp = ctx.hpart;
    double& hstep = hp[VPART];   // |q|^2 of the step under way
    unsigned* hfl = ctx.hflags + 1;

    list_rebuild(*m.nl, x, n);
    eam_gradient(e, *m.nl, d_types, d_frozen, g, FLYG_FP64);
    vec_dots(ctx, N, g, g, nullptr, nullptr, hp, hfl);
    sync_checked(ctx);
    double mag_g = host_sum(hp, 0, N);
    double trust = o.min_trust, acc = 0;
    for (int i = 0; i < o.iter_max; ++i) {
      if (iterations) *iterations = i;
      observe(ctx, m.obs, m.obs_user, i, x, n, m.obs_host);
      if (mag_g < o.f2norm * o.f2norm) return false;
      double const* qq;
      double* q = m.core->newton_step(x, g, N, nullptr, &qq, true);
      auto step = [&] { vec_step(ctx, N, trust, qq, q, x, list_move(*m.nl), m.core->stalled_word(), &hstep); };
      step();
      auto redo = [&] {   // the step gave up: x and the list are where they were
        q = m.core->again(nullptr, &qq);
        step();
      };
      // The step is at most the trust radius long: while that cannot use up the skin, its length is read
      // with the next sums instead of on its own.
      bool known = false;
      auto add_step = [&] {
        double const nrm = std::sqrt(hstep);
        double const scale = std::fmin(1.0, trust / nrm);
        acc += nrm * scale;
        known = true;
      };
      if (!(acc + 1.001 * trust < 0.5 * skin)) {
        sync(ctx);
        if (m.core->stalled()) {
          redo();
          sync(ctx);
        }
        add_step();
        if (acc > 0.5 * skin) {
          list_rebuild(*m.nl, x, n);
          acc = 0;
        }
      }
      auto look = [&] {
        eam_gradient(e, *m.nl, d_types, d_frozen, g, FLYG_FP64);
        vec_dots(ctx, N, g, q, g, g, hp, hfl);
        sync_checked(ctx);
      };
      look();
      if (m.core->stalled()) {
        redo();
        look();
      }
      if (!known) add_step();
      double proj = host_sum(hp, 0, N);
      mag_g = host_sum(hp, 1, N);
      if (proj < -o.proj_tol) {
        trust = std::fmax(o.min_trust, o.shrink_trust * trust);
      } else if (proj > o.proj_tol) {
        trust = std::fmin(o.max_trust, o.grow_trust * trust);
      }
    }
    if (iterations) *iterations = o.iter_max;
    return true;
  }

  // ================================================================================================
  // Rotor::eff_gradient (rotor.cpp:49-164) and Dimer::find_sp (dimer.cpp:28-171)
  // ================================================================================================

  namespace {

    void gradient_at(flyg_dimer_s& d, flyg_list_s& nl, flyg_eam_s& e, uint32_t const* t, uint8_t const* f, double* out) {
      eam_gradient(e, nl, t, f, out, FLYG_FP64);
      ++d.grads;
    }

  }  // namespace

  // Rotor::eff_gradient on the list nl (ready at the positions; moved by +-delta_r and back, never rebuilt).
  // Axis in/out in d.ax, effective gradient to d.eff.  Returns the curvature; |g_eff|^2 and g_eff.step (step
  // null: only the first) are left in ctx.hpart with the error flags, for the caller to read after a sync.
  // `by` (if given): the list was just moved by a step of this core; should that step have given up, *lost is set
  // and neither the list nor the axis has changed.
  double eff_gradient(flyg_dimer_s& d, flyg_list_s& nl, flyg_eam_s& e, uint32_t const* t, uint8_t const* f, long n,
                      int count_frozen, double const* step, DevLBFGS* by = nullptr, bool* lost = nullptr) {
      flyg_ctx_s& ctx = *d.ctx;
      flyg_rotor_options const& o = d.ropt;
      long N = 3 * n;
      double const dr = o.delta_r;
      d.part.reserve(2 * VPART);
      double* in = d.part.get();
      double* out = in + VPART;
      double* hp = ctx.hpart;
      double* ax = d.ax.get();
      double* g0 = d.g0.get();
      double* g1 = d.g1.get();
      double* g1p = d.g1p.get();
      double* dg = d.dg.get();
      double* dgp = d.delta_g.get();
      double* axp = d.axisp.get();
      double* dprev = d.delta_prev.get();
      ListMove const lm = list_move(nl);
      bool const none_frozen = count_frozen == 0;
      double const mean_k = -(1.0 / static_cast<double>(n));

      long const grads = d.grads;
      d.rcore->clear();
      gradient_at(d, nl, e, t, f, g0);
      rot_offset(ctx, N, dr, ax, dprev, lm, by ? by->stalled_word() : nullptr);
      gradient_at(d, nl, e, t, f, g1);
      rot_diff(ctx, N, g1, g0, ax, dg, out);

      double curv = 0;
      for (int i = 0;; ++i) {
        // Torque: delta_g = (g1 - g0) - ((g1 - g0).n) n, minus its mean when nothing is frozen; `out` holds
        // the sum (g1 - g0).n.
        std::swap(in, out);
        rot_torque(ctx, N, none_frozen, in, dg, ax, dgp, out);
        if (none_frozen) vec_demean(ctx, N, mean_k, out, dgp, nullptr, nullptr, nullptr);
        double const* thax;
        double* theta = d.rcore->newton_step(ax, dgp, N, ax, &thax, true);
        auto unit = [&] {
          rot_orth(ctx, N, thax, ax, theta, out);
          rot_unit(ctx, N, out, theta, dg, ax, hp);
          sync(ctx);
        };
        unit();
        if (i == 0 && by && by->stalled()) {
          d.grads = grads;
          *lost = true;
          return 0;
        }
        if (d.rcore->stalled()) {
          theta = d.rcore->again(ax, &thax);
          unit();
        }
        double b_1 = host_sum(hp, 0, N) / dr;
        double c_x0 = host_sum(hp, 1, N) / dr;
        double theta_1 = -0.5 * std::atan(b_1 / std::abs(c_x0));
        if (std::abs(theta_1) < o.theta_tol || (i >= o.iter_max_rot && c_x0 < 0) || i > 10 * o.iter_max_rot) {
          curv = c_x0;
          break;
        }
        // Trial rotation; the list moves from the previous end to the trial end.
        rot_trial(ctx, N, std::cos(theta_1), std::sin(theta_1), dr, ax, theta, axp, dprev, lm);
        gradient_at(d, nl, e, t, f, g1p);
        rot_curv(ctx, N, g1p, g0, axp, hp);
        sync(ctx);
        double c_x1 = host_sum(hp, 0, N) / dr;
        double a_1 = (c_x0 - c_x1 + b_1 * std::sin(2 * theta_1)) / (1 - std::cos(2 * theta_1));
        double theta_min = 0.5 * std::atan(b_1 / a_1);
        if (a_1 * std::cos(2 * theta_min) - a_1 + b_1 * std::sin(2 * theta_min) > 0) theta_min += M_PI / 2;
        double w1 = std::sin(theta_1 - theta_min) / std::sin(theta_1);
        double w2 = std::sin(theta_min) / std::sin(theta_1);
        double w3 = 1 - std::cos(theta_min) - std::sin(theta_min) * std::tan(0.5 * theta_1);
        bool const last = std::abs(theta_min) < o.theta_tol;
        rot_accept(ctx, N, std::cos(theta_min), std::sin(theta_min), w1, w2, w3, ax, theta, g1, g1p, g0, dg,
                   last ? hp : out);
        if (last) {
          sync(ctx);
          curv = host_sum(hp, 0, N) / dr;
          break;
        }
      }
      // Move the list back to the centre.
      rot_back(ctx, N, dprev, g0, ax, lm, in);
      bool const flat = !o.relax_in_convex && curv > 0;
      unsigned* hfl = ctx.hflags + 1;
      rot_eff(ctx, N, none_frozen, !flat, flat ? -1.0 : -2.0, in, g0, ax, d.eff.get(), step, none_frozen ? out : hp,
              none_frozen ? nullptr : hfl);
      if (none_frozen) vec_demean(ctx, N, mean_k, out, d.eff.get(), step, hp, hfl);
      return curv;
    }

  double rotor_eff_gradient(flyg_dimer_s& d, flyg_list_s& nl, flyg_eam_s& e, uint32_t const* t, uint8_t const* f,
                            long n, double* d_axis, double* d_eff, int count_frozen) {
    flyg_ctx_s& ctx = *d.ctx;
    require(nl.built, "List used before rebuild");
    require(nl.n == n, "rotor size mismatch");
    require(nl.rc >= e.tab.rc + 2 * d.ropt.delta_r, "the list's cut-off is below the rotor's r_cut()");
    long N = 3 * n;
    if (!d.rcore) d.rcore = std::make_unique<DevLBFGS>(&ctx, d.ropt.n, true);
    for (DVec* v : {&d.ax, &d.eff, &d.g0, &d.g1, &d.g1p, &d.dg, &d.delta_g, &d.axisp, &d.delta_prev}) v->p(N);
    copy(ctx, d.ax.get(), d_axis, N);
    double curv = eff_gradient(d, nl, e, t, f, n, count_frozen, nullptr);
    copy(ctx, d_axis, d.ax.get(), N);
    copy(ctx, d_eff, d.eff.get(), N);
    check_flags(ctx);
    return curv;
  }

  int dimer_find_sp(flyg_dimer_s& d, flyg_eam_s& e, double* d_pos, double* d_axis, uint32_t const* t,
                    uint8_t const* f, long n, double const* d_in_min, double const* d_hist, int n_hist,
                    double theta_tol, int count_frozen, flyg_search_stats* st) {
    flyg_ctx_s& ctx = *d.ctx;
    flyg_dimer_options const& o = d.opt;
    long N = 3 * n;
    double rot_rc = e.tab.rc + d.ropt.delta_r * 2;   // rotor.hpp:123
    double skin = std::fmax(std::pow(o.skin_frac, 1. / 3.) - 1, 0.0) * rot_rc;
    double rc = rot_rc + skin;
    if (!d.nl || d.nl->rc != rc) d.nl = make_list(&ctx, d.basis, d.periodic, rc);
    if (!d.core) d.core = std::make_unique<DevLBFGS>(&ctx, o.n);
    if (!d.rcore) d.rcore = std::make_unique<DevLBFGS>(&ctx, d.ropt.n, true);
    d.core->clear();
    for (DVec* v : {&d.x, &d.ax, &d.eff, &d.g0, &d.g1, &d.g1p, &d.dg, &d.delta_g, &d.axisp, &d.delta_prev, &d.tmp})
      v->p(N);
    double* hp = ctx.hpart;
    double& hstep = hp[VPART];   // |q|^2 of the step under way
    double* x = d.x.get();
    copy(ctx, x, d_pos, N);
    copy(ctx, d.ax.get(), d_axis, N);
    d.grads = 0;

    // History of known saddles, relative to the start minimum.
    std::vector<double> sn(static_cast<std::size_t>(n_hist));
    if (o.use_history && n_hist > 0) {
      if (static_cast<int>(d.hist_d.size()) < n_hist) d.hist_d.resize(static_cast<std::size_t>(n_hist));
      for (int k = 0; k < n_hist; ++k) {
        vec_diff(ctx, N, d_hist + N * k, d_in_min, d.hist_d[k].p(N), hp);
        sync(ctx);
        sn[k] = std::sqrt(host_sum(hp, 0, N));
      }
    }

    int rebuilds = 0;
    list_rebuild(*d.nl, x, n);
    double curv = eff_gradient(d, *d.nl, e, t, f, n, count_frozen, nullptr);
    sync_checked(ctx);
    double mag_g = host_sum(hp, 0, N);
    double trust = o.min_trust, acc = 0, convex_count = 0;
    int ret = FLYG_EXIT_ITER_MAX, steps = o.max_steps;
    for (int i = 0; i < o.max_steps; ++i) {
      observe(ctx, d.obs, d.obs_user, i, x, n, d.obs_host);
      if (mag_g < o.f2norm * o.f2norm) {
        ret = FLYG_EXIT_SUCCESS;
        steps = i;
        break;
      } else if (convex_count >= o.convex_max) {
        ret = FLYG_EXIT_CONVEX;
        steps = i;
        break;
      }
      if (o.use_history && n_hist > 0 && i % o.hist_check_freq == 0) {
        double* dx = d.tmp.get();
        vec_diff(ctx, N, x, d_in_min, dx, hp);
        sync(ctx);
        double on = std::sqrt(host_sum(hp, 0, N));
        double ctheta = -1;
        bool hit = false;
        for (int k = 0; k < n_hist && !hit; ++k) {
          vec_dots(ctx, N, dx, d.hist_d[k].get(), nullptr, nullptr, hp, nullptr);
          sync(ctx);
          double dt = host_sum(hp, 0, N);
          ctheta = std::fmax(ctheta, dt / (sn[k] * on));
          if (ctheta > std::cos(theta_tol)) hit = true;
        }
        if (hit) {
          ret = FLYG_EXIT_COLLISION;
          steps = i;
          break;
        }
      }
      double const* qq;
      double* q = d.core->newton_step(x, d.eff.get(), N, nullptr, &qq, true);
      auto step = [&] { vec_step(ctx, N, trust, qq, q, x, list_move(*d.nl), d.core->stalled_word(), &hstep); };
      step();
      auto redo = [&] {   // the step gave up: x and the list are where they were
        q = d.core->again(nullptr, &qq);
        step();
      };
      // As in the minimiser: the step's length is read on its own only when it could use up the skin.
      bool known = false;
      auto add_step = [&] {
        double const nrm = std::sqrt(hstep);
        double const scale = std::fmin(1.0, trust / nrm);
        acc += nrm * scale;
        known = true;
      };
      if (!(acc + 1.001 * trust < 0.5 * skin)) {
        sync(ctx);
        if (d.core->stalled()) {
          redo();
          sync(ctx);
        }
        add_step();
        if (acc > 0.5 * skin) {
          list_rebuild(*d.nl, x, n);
          acc = 0;
          ++rebuilds;
        }
      }
      bool lost = false;
      curv = eff_gradient(d, *d.nl, e, t, f, n, count_frozen, q, d.core.get(), &lost);
      if (lost) {
        redo();
        curv = eff_gradient(d, *d.nl, e, t, f, n, count_frozen, q);
      }
      convex_count = curv > 0 ? convex_count + 1 : 0;
      sync_checked(ctx);
      if (!known) add_step();
      mag_g = host_sum(hp, 0, N);
      double proj = host_sum(hp, 1, N);
      if (proj < -o.proj_tol) {
        trust = std::fmax(o.min_trust, o.shrink_trust * trust);
      } else if (proj > o.proj_tol) {
        trust = std::fmin(o.max_trust, o.grow_trust * trust);
      }
    }
    copy(ctx, d_pos, x, N);
    copy(ctx, d_axis, d.ax.get(), N);
    HIPCHK(hipStreamSynchronize(ctx.stream));
    if (st) {
      st->exit_code = ret;
      st->steps = steps;
      st->grads = d.grads;
      st->rebuilds = rebuilds;
      st->curv = curv;
      st->energy = 0;
    }
    return ret;
  }

}  // namespace flyg
