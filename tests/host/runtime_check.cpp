// Host-only checks of the library against a stand-in of the HIP runtime (runtime_stand_in.cpp): what its host code does with
// memory, streams and failed calls.  No kernel runs, so no result is looked at.  The argument picks a check.
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/pof.h"
#include "runtime_stand_in.hpp"

static int failures = 0;
#define CHECK(cond)                                                          \
  do {                                                                       \
    if (!(cond)) {                                                           \
      std::fprintf(stderr, "check failed: %s (line %d)\n", #cond, __LINE__); \
      ++failures;                                                            \
    }                                                                        \
  } while (0)

// A linear filter and smoother call of D = 12, d = 3 over n steps (device arrays: any addresses, nothing reads them)
static int filtsmooth(pof_ctx* ctx, long n, void* stream = nullptr) {
  constexpr int D = 12, d = 3;
  std::vector<double> m(D), L(D * D), F(D * D), Q(D * D);
  static double dev[1];
  double nll, obj, ssq;
  return pof_linear_filtsmooth(ctx, D, d, n, m.data(), L.data(), F.data(), Q.data(), dev, dev, nullptr, 0, nullptr, nullptr,
                               nullptr, nullptr, &nll, &obj, &ssq, stream);
}
// Steps of which a call's workspace takes about `bytes`
static long steps_for(double bytes) { return (long)(bytes / (2.0 * 8 * (7 * 144 + 7 * 12 + 2))); }

static pof_problem problem(int kind, int d, int q, std::vector<double>& ts, std::vector<double>& y0) {
  pof_problem p{};
  p.kind = kind;
  p.d = d;
  p.q = q;
  p.init = POF_INIT_CONSTANT;
  p.n_times = (int64_t)ts.size();
  p.ts_host = ts.data();
  p.y0_host = y0.data();
  p.params[0] = 8.0;
  return p;
}
static std::vector<double> grid(int n) {
  std::vector<double> ts(n);
  for (int k = 0; k < n; ++k) ts[k] = 1e-3 * k;
  return ts;
}

static int solve_large(pof_ctx* ctx, int d, int q, int n) {
  std::vector<double> ts = grid(n + 1), y0(d, 8.0);
  const pof_problem p = problem(POF_LORENZ96, d, q, ts, y0);
  pof_opts o{};
  o.maxiters = o.fixed_iters = 1;
  pof_out out{};
  return pof_solve_large(ctx, &p, &o, &out, nullptr);
}

// What calls leave for the next is given back to every other allocation of the library, of any context
static void kept_memory() {
  const double MiB = 1 << 20;
  pof_ctx *a = nullptr, *b = nullptr;
  CHECK(pof_ctx_create(0, &a) == POF_OK);
  CHECK(pof_ctx_create(0, &b) == POF_OK);
  const size_t before = stand_in::live;
  CHECK(filtsmooth(a, steps_for(400 * MiB)) == POF_OK);
  const size_t kept = stand_in::live - before;
  CHECK(kept > (size_t)(350 * MiB));
  // the next call of the context takes it
  CHECK(filtsmooth(a, steps_for(300 * MiB)) == POF_OK);
  CHECK(stand_in::live - before == kept);
  // a batch, of the other context, where nothing else is left
  stand_in::limit = stand_in::live + (size_t)(50 * MiB);
  pof_batch* batch = nullptr;
  CHECK(pof_batch_create(b, 12, 3, 2 * steps_for(200 * MiB), 1, &batch) == POF_OK);
  pof_batch_destroy(batch);
  CHECK(stand_in::live == before);
  // the large-state engine, of the other context
  stand_in::limit = ~size_t(0);
  CHECK(filtsmooth(a, steps_for(400 * MiB)) == POF_OK);
  stand_in::limit = stand_in::live + (size_t)(20 * MiB);
  CHECK(solve_large(b, 8, 2, 600) == POF_OK);
  // the linearisation's work slices
  stand_in::limit = ~size_t(0);
  CHECK(filtsmooth(a, steps_for(400 * MiB)) == POF_OK);
  stand_in::limit = stand_in::live + (size_t)(20 * MiB);
  {
    std::vector<double> ts = grid(3), y0(3, 1.0);
    const pof_problem p = problem(POF_RIGID_BODY, 3, 3, ts, y0);
    static double dev[1];
    const double par[4] = {1.0, 1.0, 0.0, 0.0};
    CHECK(pof_linearize_model(b, &p, POF_LIN_UNSCENTED, par, dev, dev, 60000, dev, dev, dev, nullptr) == POF_OK);
  }
  // a batch's launch tables and the coarse start's buffer are too small to be the ones that fail alone: that they ask
  // in the same way is in the sources (test_host_runtime.py)
  stand_in::limit = ~size_t(0);
  // an allocation that fails with nothing kept fails
  CHECK(pof_trim() >= 0 && pof_trim() == 0);
  stand_in::limit = stand_in::live + (size_t)(1 * MiB);
  CHECK(pof_batch_create(b, 12, 3, 2 * steps_for(200 * MiB), 1, &batch) == POF_E_HIP);
  stand_in::limit = ~size_t(0);
  // by hand
  const size_t base = stand_in::live;
  CHECK(filtsmooth(a, steps_for(100 * MiB)) == POF_OK);
  CHECK(filtsmooth(b, steps_for(100 * MiB)) == POF_OK);
  CHECK(stand_in::live > base + (size_t)(150 * MiB));
  CHECK(pof_trim() > (int64_t)(150 * MiB));
  CHECK(stand_in::live == base);
  pof_ctx_destroy(a);
  pof_ctx_destroy(b);
  CHECK(stand_in::live == 0);
}

// Contexts belong to threads: what all of them keep has one bound
static void kept_bound() {
  const double MiB = 1 << 20;
  std::vector<pof_ctx*> ctx(5, nullptr);
  for (auto& c : ctx) CHECK(pof_ctx_create(0, &c) == POF_OK);
  for (auto& c : ctx) {
    CHECK(filtsmooth(c, steps_for(300 * MiB)) == POF_OK);
    CHECK(filtsmooth(c, steps_for(310 * MiB)) == POF_OK);
    CHECK(stand_in::live <= (size_t)(1100 * MiB));
  }
  // one beyond the bound by itself is not kept, and takes nothing of the others'
  pof_trim();
  CHECK(filtsmooth(ctx[0], steps_for(200 * MiB)) == POF_OK);
  const size_t live = stand_in::live;
  CHECK(filtsmooth(ctx[1], steps_for(1200 * MiB)) == POF_OK);
  CHECK(stand_in::live <= live);
  // a context takes its own with it, the others' stay
  CHECK(filtsmooth(ctx[1], steps_for(200 * MiB)) == POF_OK);
  pof_ctx_destroy(ctx[0]);
  CHECK(stand_in::live > (size_t)(150 * MiB) && stand_in::live < (size_t)(250 * MiB));
  for (size_t i = 1; i < ctx.size(); ++i) pof_ctx_destroy(ctx[i]);
  CHECK(stand_in::live == 0);
}

// A call that fails once its workspace is open gives it back, and the next call has one of its own
static void failed_call() {
  pof_ctx* ctx = nullptr;
  CHECK(pof_ctx_create(0, &ctx) == POF_OK);
  const size_t before = stand_in::live;
  for (const char* kernel : {"k_upload", "k_filter_leaf16", "k_filter_up16", "k_reduce_final", "k_output"}) {
    CHECK(filtsmooth(ctx, 100) == POF_OK);
    CHECK(stand_in::live > before);
    stand_in::fail_launch = kernel;
    CHECK(filtsmooth(ctx, 90) == POF_E_HIP);
    CHECK(stand_in::fail_launch.empty());
    CHECK(stand_in::live == before);
    CHECK(filtsmooth(ctx, 90) == POF_OK);
    pof_trim();
  }
  pof_ctx_destroy(ctx);
  CHECK(stand_in::live == 0);
}

// The words that launches of k_upload bring to the device (its argument: {source, destination, words} per grid row)
static size_t g_words = 0;
static void count_words(const std::string& name, unsigned rows, void** args) {
  struct Part {
    const unsigned* src;
    unsigned* dst;
    size_t n;
  };
  if (name.find("k_upload") == std::string::npos) return;
  const Part* p = static_cast<const Part*>(args[0]);
  for (unsigned i = 0; i < rows; ++i) g_words += p[i].n;
}

// A batch after a call that failed part way: its tables are not taken to be on the device, and the host's are not
// written while an upload may still be reading them
static void failed_launch() {
  pof_ctx* ctx = nullptr;
  CHECK(pof_ctx_create(0, &ctx) == POF_OK);
  pof_batch* b = nullptr;
  CHECK(pof_batch_create(ctx, 12, 3, 4096, 4, &b) == POF_OK);
  stand_in::on_launch = count_words;
  std::vector<double> ts = grid(65), y0(3, 1.0);
  const pof_problem p = problem(POF_RIGID_BODY, 3, 3, ts, y0);
  pof_opts o{};
  o.maxiters = o.fixed_iters = 2;
  pof_out out[4] = {};
  for (int i = 0; i < 2; ++i) CHECK(pof_batch_admit(b, &p, &o, &out[i], nullptr) == POF_OK);
  // the upload of an admission
  stand_in::fail_launch = "k_upload";
  g_words = 0;
  CHECK(pof_batch_launch(b) == POF_E_HIP);
  const size_t first = g_words;
  g_words = 0;
  // ... and, once it has gone, a launch behind it
  stand_in::fail_launch = "k_filter_leaf16";
  CHECK(pof_batch_launch(b) == POF_E_HIP);
  CHECK(first > 0 && g_words == first);
  const long syncs = stand_in::syncs;
  CHECK(pof_batch_admit(b, &p, &o, &out[2], nullptr) == POF_OK);
  CHECK(stand_in::syncs > syncs);
  // two iterations, and a retirement that fails
  CHECK(pof_batch_launch(b) == POF_OK);
  int n = 0;
  CHECK(pof_batch_finish(b, 0, nullptr, &n) == POF_OK && n == 0);
  g_words = 0;
  CHECK(pof_batch_launch(b) == POF_OK);
  CHECK(g_words == 4);  // the factor flags of the last iteration alone
  stand_in::fail_launch = "k_output";
  CHECK(pof_batch_finish(b, 0, nullptr, &n) == POF_E_HIP);
  g_words = 0;
  CHECK(pof_batch_launch(b) == POF_OK);
  CHECK(g_words >= 3 * 4);  // the launch tables (records of three IVPs, ...), which the retirement's have overwritten
  stand_in::on_launch = nullptr;
  pof_batch_destroy(b);
  pof_ctx_destroy(ctx);
  CHECK(stand_in::live == 0);
}

// More parts than one upload launch takes, the first of whose launches fails: the others go nowhere, and the retry has all
static void failed_upload_of_many() {
  pof_ctx* ctx = nullptr;
  CHECK(pof_ctx_create(0, &ctx) == POF_OK);
  constexpr int kIvps = 60;
  pof_batch* b = nullptr;
  CHECK(pof_batch_create(ctx, 12, 3, 4096, kIvps, &b) == POF_OK);
  stand_in::on_launch = count_words;
  std::vector<double> ts = grid(5), y0(3, 1.0);
  pof_problem p = problem(POF_RIGID_BODY, 3, 3, ts, y0);
  p.init = POF_INIT_PRIOR;  // initial means from the host: a part each
  pof_opts o{};
  o.maxiters = o.fixed_iters = 2;
  std::vector<pof_out> out(kIvps);
  for (auto& x : out) CHECK(pof_batch_admit(b, &p, &o, &x, nullptr) == POF_OK);
  stand_in::fail_launch = "k_upload";
  CHECK(pof_batch_launch(b) == POF_E_HIP);
  g_words = 0;
  CHECK(pof_batch_launch(b) == POF_OK);
  CHECK(g_words > (size_t)kIvps * 5 * 12 * 2);
  stand_in::on_launch = nullptr;
  pof_batch_destroy(b);
  pof_ctx_destroy(ctx);
  CHECK(stand_in::live == 0);
}

// A call on a stream that its caller is capturing is refused before anything is enqueued: what it enqueued would
// stay in the caller's graph, over memory that the refused call gives back
static void captured_stream() {
  pof_ctx* ctx = nullptr;
  CHECK(pof_ctx_create(0, &ctx) == POF_OK);
  int handle = 0;
  void* stream = &handle;
  std::vector<double> ts = grid(65), y0(3, 1.0), m(12), L(144), F(144), Q(144);
  const pof_problem p = problem(POF_RIGID_BODY, 3, 3, ts, y0);
  pof_opts o{};
  o.maxiters = o.fixed_iters = 2;
  pof_out out{};
  std::vector<double> dev(64 * 1024);
  double nll, obj, ssq;
  auto call = [&](int k) {
    switch (k) {
      case 0: return filtsmooth(ctx, 64, stream);
      case 1: return pof_solve(ctx, &p, &o, &out, stream);
      case 2: return pof_eks_solve(ctx, &p, 1, &out, stream);
      case 3: return pof_ieks_step(ctx, &p, dev.data(), 0, nullptr, nullptr, &nll, &obj, &ssq, stream);
      case 4: return pof_smoothing(ctx, 12, 64, F.data(), Q.data(), dev.data(), dev.data(), 0, nullptr, nullptr, &obj, stream);
      default: return pof_ekf(ctx, &p, m.data(), L.data(), F.data(), Q.data(), nullptr, nullptr, &nll, &ssq, stream);
    }
  };
  for (int warm = 0; warm < 2; ++warm) {  // without and with workspaces of calls before
    for (int k = 0; k < 6; ++k) {
      const long n = stand_in::launched("");
      const size_t live = stand_in::live;
      stand_in::capturing = stream;
      CHECK(call(k) == POF_E_HIP);
      CHECK(std::strlen(pof_last_error(ctx)) > 0);
      stand_in::capturing = nullptr;
      CHECK(stand_in::launched("") == n);
      CHECK(stand_in::live == live);
      CHECK(call(k) == POF_OK);
      CHECK(stand_in::launched("") > n);
    }
  }
  pof_ctx_destroy(ctx);
  CHECK(stand_in::live == 0);
}

// The large-state engine over every shape that it takes (a grid of the longest there is among them): its workspace is large
// enough, and every kernel of the factorisation that the library holds is one that some shape runs
static void large_shapes() {
  int shapes = 0;
  for (int d = 1; d <= 4; ++d)  // fields of the per-worker kernels, whose states the engine takes too
    for (int q = 1; q <= 5; ++q) {
      if (!pof_supported(d * (q + 1), d)) continue;
      const int kinds[] = {POF_LOGISTIC, POF_FHN_CLASSIC, POF_RIGID_BODY, POF_HENONHEILES};
      for (int n : {1, 2, 3, 7, 64, 1025, 4099}) {
        std::vector<double> ts = grid(n + 1), y0(d, 0.5);
        const pof_problem p = problem(kinds[d - 1], d, q, ts, y0);
        pof_opts o{};
        o.maxiters = o.fixed_iters = 1;
        pof_out out{};
        pof_ctx* c = nullptr;
        CHECK(pof_ctx_create(0, &c) == POF_OK);
        CHECK(pof_solve_large(c, &p, &o, &out, nullptr) == POF_OK);
        pof_ctx_destroy(c);
      }
    }
  for (int d = 4; d <= 64; ++d)
    for (int q = 1; d * (q + 1) <= 128; ++q) {
      std::vector<double> ts = grid(3), y0(d, 8.0);
      const pof_problem p = problem(POF_LORENZ96, d, q, ts, y0);
      if (pof_setup(&p, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr) != POF_OK) continue;
      ++shapes;
      for (int n : {1, 2, 3, 5, 6, 7, 11, 64, 65, 200, 1025, 2047, 2048, 4099, 65534}) {
        if (n > 5000 && q > 3) continue;
        // a fresh context for each: the engine's buffer grows and is not given back
        pof_ctx* c = nullptr;
        CHECK(pof_ctx_create(0, &c) == POF_OK);
        const int rc = solve_large(c, d, q, n);
        if (rc != POF_OK) std::fprintf(stderr, "d=%d q=%d n=%d: %s\n", d, q, n, pof_last_error(c));
        CHECK(rc == POF_OK);
        pof_ctx_destroy(c);
      }
    }
  CHECK(shapes > 40);
  for (const std::string& k : stand_in::kernels("k_lq_")) {
    if (stand_in::launched(k) == 0) std::fprintf(stderr, "not reached: %s\n", k.c_str());
    CHECK(stand_in::launched(k) > 0);
  }
  CHECK(stand_in::live == 0);
}

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "kept_memory") kept_memory();
  else if (what == "kept_bound") kept_bound();
  else if (what == "failed_launch") failed_launch();
  else if (what == "captured_stream") captured_stream();
  else if (what == "large_shapes") large_shapes();
  else if (what == "failed_call") failed_call();
  else if (what == "failed_upload_of_many") failed_upload_of_many();
  else CHECK(!"a known check");
  std::printf("%s: %d failures\n", what.c_str(), failures);
  return failures == 0 ? 0 : 1;
}
