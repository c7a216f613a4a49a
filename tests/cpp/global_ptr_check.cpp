// The contract of global_ptr (csrc/de_common.h) on the host: no lane passes it an
// address of its own stack.  Every pointer it is given is checked while the event
// lanes integrate (deferred brackets, t_eval output), run the root and bookkeeping
// passes over the brackets, and solve the same trajectories with inline roots.
// Prints the brackets rooted and, per lane, the stack pointers seen.
#include <pthread.h>
#include <stdio.h>

#include <vector>

static const char *g_lo, *g_hi;
static long g_stack, g_seen;
static void on_global_ptr(const volatile void* p) {
  ++g_seen;
  if ((const char*)p >= g_lo && (const char*)p < g_hi) ++g_stack;
}
#define DE_ON_GLOBAL_PTR(p) ::on_global_ptr(p)
#include "../../differential-equations_amd/csrc/de_erk_lane.h"

using namespace de;

static long g_brackets;
static int g_bad;

template <class Lane>
static void run(const char* name, int solout, int fn, int n_eval) {
  constexpr int D = Lane::D, n = 5, bmax = 64, max_events = 16;
  std::vector<double> params = {10, 9, 11, 10, 10.5, 28, 29, 27, 30, 28, 2.5, 2.6, 2.7, 2.6, 2.5};
  std::vector<double> y0(n * D), t0(n, 0.0), tf(n, 3.0), rt(n, 1e-6), at(n, 1e-9);
  std::vector<double> rc(n * D, 1e-6), ac(n * D, 1e-9), te, value(n, 0.3);
  for (int i = 0; i < n * D; ++i) y0[i] = 1.0 + 0.37 * i;
  for (int e = 0; e < n_eval; ++e) te.push_back(0.1 + 0.25 * e);
  std::vector<double> y(n * D), t(n), dense(n * D * (n_eval + 1)), point(D, 1.0), normal(D, 1.0);
  std::vector<int64_t> acc(n), rej(n), ev(n);
  std::vector<int32_t> status(n), nd(n), bcount(n), n_out(n);
  std::vector<double> brk((size_t)n * bmax * Lane::kEntryWidth), res((size_t)n * bmax * kResWidth);
  std::vector<double> ev_t(n * max_events), ev_y(n * max_events * D);
  OdeArgs a = {};
  a.n = n;
  a.params = params.data();
  a.y0 = y0.data();
  a.t0 = t0.data();
  a.tf = tf.data();
  a.rtol_traj = rt.data();
  a.atol_traj = at.data();
  a.rtol_comp = rc.data();
  a.atol_comp = ac.data();
  a.h0 = 0.01;
  a.h_max = 0.1;
  a.safety = 0.9;
  a.min_scale = 0.2;
  a.max_scale = 10.0;
  a.max_steps = 5000;
  a.max_rejects = 100;
  a.t_eval = te.data();
  a.n_eval = n_eval;
  a.y_final = y.data();
  a.t_final = t.data();
  a.accepted = acc.data();
  a.rejected = rej.data();
  a.evals = ev.data();
  a.status = status.data();
  a.dense = dense.data();
  a.n_dense = n_eval ? nd.data() : nullptr;
  a.ev.solout = solout;
  a.ev.fn = fn;
  a.ev.max_events = max_events;
  a.ev.value_traj = value.data();
  a.ev.point = point.data();
  a.ev.normal = normal.data();
  a.ev.t_out = ev_t.data();
  a.ev.y_out = ev_y.data();
  a.ev.n_out = n_out.data();
  a.ev.brk = brk.data();
  a.ev.res = res.data();
  a.ev.bcount = bcount.data();
  a.ev.bmax = bmax;
  a.ev.width = Lane::kEntryWidth;
  const long stack0 = g_stack;
  long rooted = 0;
  for (int inline_roots = 0; inline_roots < 2; ++inline_roots) {
    if (inline_roots) a.ev.brk = nullptr;
    for (int i = 0; i < n; ++i) {
      Lane::predicted_cost(a, i);
      Lane L;
      if (L.begin(a, i))
        while (!L.advance(a, i)) {
        }
      if (inline_roots) continue;
      for (int k = 0; k < bcount[i]; ++k, ++rooted) {
        const int64_t slot = (int64_t)i * bmax + k;
        Lane::entry_root(a, i, a.ev.brk + slot * a.ev.width, a.ev.res + slot * kResWidth);
      }
      Lane::entry_book(a, i);
    }
  }
  if (g_stack != stack0 || rooted == 0) g_bad = 1;
  printf("%s solout %d fn %d t_eval %d: %ld brackets, %ld stack pointers\n", name, solout, fn,
         n_eval, rooted, g_stack - stack0);
  g_brackets += rooted;
}

int main() {
  pthread_attr_t attr;
  void* base;
  size_t size;
  pthread_getattr_np(pthread_self(), &attr);
  pthread_attr_getstack(&attr, &base, &size);
  g_lo = (const char*)base;
  g_hi = g_lo + size;
  using F = LorenzRhs;
  using namespace erk_tab;
#define DE_RUN(NAME, LANE1, LANE2)                            \
  run<LANE1>(NAME, kSoloutEvent, kEventComponent, 0);         \
  run<LANE1>(NAME, kSoloutEvent, kEventPlane, 7);             \
  run<LANE2>(NAME, kSoloutCrossing, kEventComponent, 0);      \
  run<LANE2>(NAME, kSoloutHyperplane, kEventPlane, 0);
  using D5a = Dopri5Lane<F, true, true, 1>;
  using D5b = Dopri5Lane<F, false, false, 2>;
  using D8a = Dop853Lane<F, true, true, 1>;
  using D8b = Dop853Lane<F, false, false, 2>;
  using R4a = FixedLane<F, 4, 1>;
  using R4b = FixedLane<F, 4, 2>;
  using E1a = FixedLane<F, 1, 1>;
  using E1b = FixedLane<F, 1, 2>;
  using K4a = ErkLane<F, Rkf45, true, true, 1>;
  using K4b = ErkLane<F, Rkf45, false, true, 2>;
  using V7a = ErkLane<F, Rkv767e, true, true, 1>;
  using V7b = ErkLane<F, Rkv767e, false, true, 2>;
  DE_RUN("dopri5", D5a, D5b)
  DE_RUN("dop853", D8a, D8b)
  DE_RUN("rk4", R4a, R4b)
  DE_RUN("euler", E1a, E1b)
  DE_RUN("rkf45", K4a, K4b)
  DE_RUN("rkv767e", V7a, V7b)
  printf("%ld pointers checked\n", g_seen);
  return g_bad;
}
